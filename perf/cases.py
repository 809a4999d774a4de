"""Performance cases: the work that programs give this framework, through its public entry points.

Three kinds.  ``decoder``: the quantized decoder (Q4_0 attention and tables, TQ2_0 feed-forward, 2-bit keys and values) through
``generation.PipelineSequences`` and ``DecodePipeline.decode_batch_step``.  ``stack``: models with bf16 weights through
``StackPipeline``, a request at a time as a trace replay runs it: a sequence is opened, its prompt fed in portions, then its
tokens one by one, and the sequence is closed.  ``matvec``, ``matmul`` and ``attention``: single dispatches of ``Kernels``, for
programs that drive the operators themselves.

``exact`` states every kind in 64 bits with plain torch."""
import math
import os
import sys

import numpy as np
import torch

if os.getcwd() not in sys.path:
    sys.path.insert(0, os.getcwd())
from __graft_entry__ import load_package  # noqa: E402

pkg = load_package()
DEVICE = "cuda"
F64 = torch.float64
_context = []


def context():
    """The program's one device context and its kernels."""
    if not _context:
        ctx = pkg.Context(0)
        _context.extend((ctx, pkg.Kernels(ctx)))
    return _context


# ---- the cases ----------------------------------------------------------------------------------------------------------
def listed():
    e2b = {"kind": "decoder", "hidden": 1536, "layers": 10, "ff": 6144, "vocab": 262144}
    komirax = {"kind": "stack", "design": "Komirax", "vocab": 32000}
    vifivik = {"kind": "stack", "design": "Vifivik", "vocab": 32000}
    return [
        # one generated token of a chat with a long history: latency, a launch after the other
        {"name": "quantized token", **e2b, "mode": "token", "context": 32768, "rows": 1},
        # a server's step: one token for each of its live sequences, which are not equally long
        {"name": "quantized step of 64", **e2b, "mode": "lanes", "context": 16384, "rows": 64},
        # the end of a long prompt: a chunk of the largest size and the token whose logits are sampled
        {"name": "quantized prompt chunk", **e2b, "mode": "prompt", "context": 16000, "rows": 257},
        # a whole long prompt, in the largest passes
        {"name": "prompt of 4096", **komirax, "width": 2048, "prompt": 4096, "new": 0, "portion": 4096, "dtype": "bf16"},
        {"name": "latent prompt of 3001", **vifivik, "width": 2048, "prompt": 3001, "new": 0, "portion": 3001, "dtype": "bf16"},
        # a prompt in the scheduler's default portions, of a smaller model; the last portion is ragged
        {"name": "prompt in portions", **komirax, "width": 1024, "prompt": 1700, "new": 0, "portion": 512, "dtype": "bf16"},
        # answers: a short question and the tokens that follow it
        {"name": "answer of 48", **komirax, "width": 2048, "prompt": 200, "new": 48, "portion": 512, "dtype": "bf16"},
        {"name": "latent answer of 48", **vifivik, "width": 1024, "prompt": 200, "new": 48, "portion": 512, "dtype": "bf16"},
        # a reference run in 32 bits, as a trace replay with --dtype float32 makes it
        {"name": "replay in 32 bits", **komirax, "width": 1024, "prompt": 333, "new": 4, "portion": 333, "dtype": "f32"},
        # a stack of projections, one vector each: weight streaming
        {"name": "rows of weights", "kind": "matvec", "format": "tq2_0", "rows": 8192, "cols": 2048, "count": 128},
        # a prompt's feed-forward product
        {"name": "prompt product", "kind": "matmul", "format": "q4_0", "m": 512, "k": 2048, "n": 8192, "input": "bf16", "output": "f32"},
        # attention over the 2-bit caches of many sequences
        {"name": "code attention", "kind": "attention", "context": 32768, "lanes": 128, "head_dim": 256, "window": 0},
    ]


def spread(rng, lo, hi):
    """A whole number from lo to hi, evenly over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decoder", "decoder", "decoder", "stack", "stack", "stack", "stack", "matvec", "matmul", "attention"])
    if kind == "decoder":
        mode = rng.choice(["token", "lanes", "prompt"])
        rows = {"token": 1, "lanes": spread(rng, 2, 64), "prompt": spread(rng, 17, 257)}[mode]
        return {"kind": kind, "mode": mode, "hidden": 256 * rng.randint(4, 8), "layers": rng.randint(5, 10), "ff": 256 * rng.randint(16, 24),
                "vocab": spread(rng, 32000, 262144), "context": spread(rng, 700, 32768 if mode == "token" else 16384), "rows": rows}
    if kind == "stack":
        design, part = rng.choice(["Komirax", "Vifivik"]), rng.choice(["prompt", "prompt", "portions", "answer", "answer", "f32"])
        c = {"kind": kind, "design": design, "vocab": spread(rng, 8000, 32000), "width": 128 * rng.randint(8, 16), "new": 0, "dtype": "bf16"}
        if part == "prompt":
            c["prompt"] = c["portion"] = spread(rng, 65, 4000)
        elif part == "portions":
            c.update(prompt=spread(rng, 600, 2000), portion=rng.randint(256, 512))
        elif part == "answer":
            c.update(prompt=spread(rng, 16, 1000), portion=512, new=spread(rng, 8, 48))
        else:
            c.update(prompt=spread(rng, 20, 333), new=rng.randint(0, 4), portion=333, dtype="f32", width=128 * rng.randint(6, 8))
        return c
    if kind == "matvec":
        cols = rng.choice([1536, 2048, 2048, 4096, 6144, 8192])
        return {"kind": kind, "format": rng.choice(["tq2_0", "q4_0"]), "rows": spread(rng, 256, 8192), "cols": cols, "count": rng.randint(1, 48)}
    if kind == "matmul":
        return {"kind": kind, "format": rng.choice(["tq2_0", "q4_0"]), "m": spread(rng, 65, 512), "k": 256 * rng.randint(6, 12),
                "n": 64 * rng.randint(32, 128), "input": rng.choice(["bf16", "f16"]), "output": rng.choice(["f32", "f16"])}
    window = rng.choice([0, 0, 512])
    return {"kind": kind, "context": 64 * spread(rng, 16, 512), "lanes": spread(rng, 1, 128), "head_dim": 256, "window": window}


# ---- seeded inputs ------------------------------------------------------------------------------------------------------
class Source:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEVICE)

    def whole(self, below, *shape):
        return torch.randint(0, below, shape, generator=self.g, device=DEVICE)

    def order(self, n, count):
        return torch.rand(count, n, generator=self.g, device=DEVICE).argsort(1)

    def bytes(self, *shape):
        return self.whole(256, *shape).to(torch.uint8)

    def blocks(self, fmt, rows, cols):
        """A packed matrix: Q4_0 [rows, cols / 32, 18] or TQ2_0 [rows, cols / 256, 66] bytes."""
        if fmt == "q4_0":
            d = (self.normal(rows, cols // 32, 1).abs() * (0.02 / 8)).half()
            return torch.cat([d.view(torch.uint8), self.bytes(rows, cols // 32, 16)], 2)
        code = (self.whole(81, rows, cols // 256, 64)).to(torch.int16)         # four digits of 0, 1 or 2
        code = code % 3 | code // 3 % 3 << 2 | code // 9 % 3 << 4 | code // 27 << 6
        d = (self.normal(rows, cols // 256, 1).abs() * 0.02).half()
        return torch.cat([code.to(torch.uint8), d.view(torch.uint8)], 2)


def unpack(raw):
    """A packed matrix as float64 [rows, cols]."""
    if raw.shape[2] == 18:
        d, q = raw[..., :2].contiguous().view(torch.float16).to(F64), raw[..., 2:]
        return ((torch.cat([q & 15, q >> 4], 2).to(F64) - 8) * d).flatten(1)
    d, q = raw[..., 64:].contiguous().view(torch.float16).to(F64), raw[..., :64].unflatten(2, (2, 1, 32))
    code = torch.cat([q >> 2 * i & 3 for i in range(4)], 3)
    return ((code.flatten(2).to(F64) - 1) * d).flatten(1)


def upload(t):
    """A buffer of the framework's own that holds the tensor."""
    ctx, _ = context()
    t = t.contiguous()
    torch.cuda.synchronize()
    nbytes = t.numel() * t.element_size()
    b, batch = pkg.Buffer.empty(ctx, nbytes), pkg.CommandBatch(ctx)
    batch.blit_copy(pkg.Buffer.wrap(ctx, t.data_ptr(), nbytes), 0, b, 0, nbytes)
    batch.commit_and_wait()
    return b


def wrap(t):
    return pkg.Buffer.wrap(context()[0], t.data_ptr(), t.numel() * t.element_size(), owner=t)


def on_device(a):
    return torch.from_numpy(np.array(a)).to(DEVICE)


FORMAT = {"q4_0": pkg.Q4_0, "tq2_0": pkg.TQ2_0}
TYPE = {"bf16": (pkg.BF16, torch.bfloat16), "f16": (pkg.F16, torch.float16), "f32": (pkg.F32, torch.float32)}


# ---- the quantized decoder ----------------------------------------------------------------------------------------------
HEADS, PER_LAYER, WINDOW, EPS = 8, 256, 512, 1e-6


def decoder_config(c):
    n = c["layers"]
    return pkg.pipeline.Gemma4QATConfig(
        vocab_size=c["vocab"], hidden_size=c["hidden"], num_hidden_layers=n, num_attention_heads=HEADS, num_key_value_heads=1, head_dim=256,
        global_head_dim=512, sliding_window=WINDOW, num_kv_shared_layers=n - 5, hidden_size_per_layer_input=PER_LAYER,
        layer_types=["full_attention" if i % 5 == 4 else "sliding_attention" for i in range(n)], sliding_rope_theta=10000.0,
        full_rope_theta=1000000.0, full_partial_rotary_factor=0.25)


def decoder_shapes(c, cfg, i):
    """name -> (format, rows, columns) of layer i's projections: the layers that read another's cache are twice as wide."""
    h, hd, ff = c["hidden"], cfg.attn_head_dim(i), c["ff"] * (2 if cfg.is_kv_shared(i) else 1)
    s = {"attn_q": ("q4_0", HEADS * hd, h), "attn_output": ("q4_0", h, HEADS * hd), "ffn_gate": ("tq2_0", ff, h), "ffn_up": ("tq2_0", ff, h),
         "ffn_down": ("tq2_0", h, ff), "per_layer_inp_gate": ("q4_0", PER_LAYER, h), "per_layer_proj": ("q4_0", h, PER_LAYER)}
    if not cfg.is_kv_shared(i):
        s.update(attn_k=("q4_0", hd, h), attn_v=("q4_0", hd, h))
    return s


def decoder_inputs(c, seed):
    """Every tensor of the model, the tokens and positions; what stands in the caches comes from `decoder_cache`."""
    cfg, src = decoder_config(c), Source(seed)
    h, n = c["hidden"], c["layers"]

    def norm(k, mean=1.0):
        return ((1 + 0.1 * src.normal(k)) * mean).half()
    layers = []
    for i in range(n):
        hd = cfg.attn_head_dim(i)
        t = {name: src.blocks(*s) for name, s in decoder_shapes(c, cfg, i).items()}
        t.update({name: norm(h) for name in ("attn_norm", "attn_post_norm", "ffn_norm", "ffn_post_norm", "per_layer_post_norm")})
        t["q_norm"] = norm(hd, hd ** -0.25)              # scores of about unit spread
        if not cfg.is_kv_shared(i):
            t["k_norm"] = norm(hd, hd ** -0.25)
        layers.append(t)
    rows = c["rows"]
    m = {"layers": layers, "embed": src.blocks("q4_0", c["vocab"], h), "table": src.blocks("q4_0", c["vocab"], n * PER_LAYER),
         "model_proj": src.blocks("q4_0", n * PER_LAYER, h), "proj_norm": norm(PER_LAYER), "output_norm": norm(h),
         "tokens": src.whole(c["vocab"], rows).tolist()}
    m["positions"] = [c["context"]] * rows
    if c["mode"] == "lanes":
        m["positions"] = [c["context"] // 2 + v for v in src.whole(c["context"] - c["context"] // 2, rows).tolist()]
    return cfg, m, src


def decoder_prepare(c, seed):
    ctx, K = context()
    cfg, m, src = decoder_inputs(c, seed)
    lanes, T = c["mode"] == "lanes", c["context"]
    P, L = pkg.pipeline, pkg.layer

    def weight(raw, fmt="q4_0"):
        cols = raw.shape[1] * (32 if fmt == "q4_0" else 256)
        return pkg.QuantWeight.quantized(upload(raw), FORMAT[fmt], raw.shape[0], cols)
    layers = []
    for i, t in enumerate(m["layers"]):
        shapes = decoder_shapes(c, cfg, i)
        w = L.LayerWeights(**{name: weight(x, shapes[name][0]) if name in shapes else upload(x) for name, x in t.items()})
        full = cfg.is_full_attention(i)
        layers.append(L.TransformerLayer(L.LayerParams(
            layer_idx=i, hidden_size=c["hidden"], intermediate_size=w.ffn_gate.rows, num_attention_heads=HEADS, num_key_value_heads=1,
            head_dim=cfg.attn_head_dim(i), per_layer_dim=PER_LAYER, rope_theta=cfg.rope_theta(i), partial_rotary_factor=cfg.partial_rotary_factor(i),
            sliding_window=0 if full else WINDOW, rms_norm_eps=EPS, is_kv_shared=cfg.is_kv_shared(i)), w))
    embed, table = weight(m["embed"]), weight(m["table"])
    pipe = P.DecodePipeline(ctx, K, cfg, layers, embed, upload(m["output_norm"]), T + 512 if not lanes else 2048,
                            pkg.weights.QuantRowTable(table, pkg.gguf.GGUFType.Q4_0, table.device_bytes()), weight(m["model_proj"]),
                            upload(m["proj_norm"]))
    s = {"case": c, "pipe": pipe, "tokens": m["tokens"], "positions": m["positions"]}
    if lanes:
        state = pipe.new_batched_decode_state(c["rows"], max(T + 64, 1024))
        s["logits"] = torch.empty(c["rows"], c["vocab"], device=DEVICE)      # sampled on the device
        state.logits_buf = wrap(s["logits"])
        s["state"], caches = state, state.pools
    else:
        s["model"], caches = pkg.generation.PipelineSequences(pipe), pipe.kv_caches
        s["seq"] = s["model"].new_sequence()
    for cache in caches:                                   # what the tokens before have left there
        n = (cache.lane_stride() * cache.n_lanes) if lanes else cache.physical_positions
        for codes, norms, scale in ((cache.keys_q, cache.key_norms, cache.head_dim ** -0.25), (cache.values_q, cache.value_norms, 1.0)):
            for lo in range(0, n, 1 << 19):
                count = min(n - lo, 1 << 19)
                rows = (src.normal(count, cache.head_dim) * scale).half()
                torch.cuda.synchronize()
                batch = pkg.CommandBatch(ctx)
                K.encode_kv_turboquant_into(batch, wrap(rows), cache.levels, cache.signs, codes, norms, cache.head_dim, 1, count, cache.bits, lo, 0)
                batch.commit_and_wait()
    return s


def decoder_run(s):
    c = s["case"]
    if c["mode"] == "lanes":
        s["pipe"].decode_batch_step(s["state"], s["tokens"], s["tokens"], s["positions"], read_logits=False)
        return s["logits"]
    s["pipe"].position = c["context"]
    return s["model"].step(s["seq"], s["tokens"], [len(s["tokens"]) - 1])


def unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def hadamard(x):
    n = x.shape[-1]
    y = x.reshape(-1, n)
    step = 1
    while step < n:
        y = y.reshape(-1, n // (2 * step), 2, step)
        y = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], 2)
        step *= 2
    return y.reshape(x.shape) / math.sqrt(n)


def code_values(codes, norms, levels, count, hd):
    """Cache rows in rotated space, float64 [count, hd]."""
    b = on_device(codes.as_array(np.uint8, count * hd // 4)).reshape(count, hd // 4, 1)
    code = torch.cat([b >> 2 * i & 3 for i in range(4)], 2).reshape(count, hd)
    return levels[code.long()] * on_device(norms.as_array(np.float16, count)).to(F64)[:, None]


def decoder_exact(c, seed):
    s = decoder_prepare(c, seed)
    cfg, m, _ = decoder_inputs(c, seed)
    lanes, T, R, h = c["mode"] == "lanes", c["context"], c["rows"], c["hidden"]
    caches = s["state"].pools if lanes else s["pipe"].kv_caches
    pos = torch.tensor(m["positions"], device=DEVICE) + (0 if lanes else torch.arange(R, device=DEVICE))
    past = []
    for cache in caches:
        n = cache.lane_stride() * cache.n_lanes if lanes else cache.physical_positions
        levels, signs = on_device(cache.levels.as_array(np.float32)).to(F64), on_device(cache.signs.as_array(np.float32)).to(F64)
        ring = cache.lane_ring_capacity if lanes else cache.ring_capacity()
        past.append((levels, signs, ring, code_values(cache.keys_q, cache.key_norms, levels, n, cache.head_dim),
                     code_values(cache.values_q, cache.value_norms, levels, n, cache.head_dim)))

    def rope(x, hd, theta, part):                            # x [R, heads, hd]
        k = int(hd * part) // 2
        a = pos[:, None].to(F64) * theta ** (-2.0 * torch.arange(k, device=DEVICE, dtype=F64) / hd)
        u, v, y = x[..., :k], x[..., hd // 2:hd // 2 + k], x.clone()
        y[..., :k], y[..., hd // 2:hd // 2 + k] = u * a.cos()[:, None] - v * a.sin()[:, None], u * a.sin()[:, None] + v * a.cos()[:, None]
        return y

    def encoded(x, levels, signs):
        n = x.half().to(F64).norm(dim=1, keepdim=True)
        y = hadamard(x / n * signs)
        return levels[(y[..., None] - levels).abs().argmin(-1)] * n.half().to(F64)
    tokens = torch.tensor(m["tokens"], device=DEVICE)
    x = unpack(m["embed"][tokens]) * math.sqrt(h)
    proj = (x @ unpack(m["model_proj"]).T / math.sqrt(h)).reshape(R, -1, PER_LAYER)
    ple = (unit(proj, EPS) * m["proj_norm"].to(F64) + unpack(m["table"][tokens]).reshape(proj.shape) * math.sqrt(PER_LAYER)) * math.sqrt(0.5)
    for i, t in enumerate(m["layers"]):
        w = {name: unpack(v) if v.dim() == 3 else v.to(F64) for name, v in t.items()}
        hd, theta, part, full = cfg.attn_head_dim(i), cfg.rope_theta(i), cfg.partial_rotary_factor(i), cfg.is_full_attention(i)
        slot = s["pipe"].kv_index_map[i]
        levels, signs, ring, kc, vc = past[slot]
        y = unit(x, EPS) * w["attn_norm"]
        q = rope(unit((y @ w["attn_q"].T).reshape(R, HEADS, hd), EPS) * w["q_norm"], hd, theta, part)
        if "attn_k" in w:
            k = rope((unit(y @ w["attn_k"].T, EPS) * w["k_norm"])[:, None], hd, theta, part)[:, 0]
            at = (pos % ring if ring else pos) + (torch.arange(R, device=DEVICE) * caches[slot].lane_stride() if lanes else 0)
            kc[at], vc[at] = encoded(k, levels, signs), encoded(unit(y @ w["attn_v"].T, EPS), levels, signs)
        q = hadamard(q * signs)
        o = torch.empty_like(q)
        for lo in range(0, R, 1 if lanes else 32):
            hi = lo + 1 if lanes else min(lo + 32, R)
            last = int(pos[hi - 1])
            first = 0 if full else max(0, int(pos[lo]) + 1 - WINDOW)
            p = torch.arange(first, last + 1, device=DEVICE)
            at = (p % ring if ring else p) + (lo * caches[slot].lane_stride() if lanes else 0)
            seen = p[None] <= pos[lo:hi, None]
            if not full:
                seen &= p[None] > pos[lo:hi, None] - WINDOW
            z = (q[lo:hi] @ kc[at].T).masked_fill(~seen[:, None], -math.inf)
            o[lo:hi] = torch.softmax(z, -1) @ vc[at]
        o = (hadamard(o) * signs).reshape(R, -1)
        x = x + unit(o @ w["attn_output"].T, EPS) * w["attn_post_norm"]
        y = unit(x, EPS) * w["ffn_norm"]
        y = (gelu_tanh(y @ w["ffn_gate"].T) * (y @ w["ffn_up"].T)) @ w["ffn_down"].T
        x = x + unit(y, EPS) * w["ffn_post_norm"]
        y = (gelu_tanh(x @ w["per_layer_inp_gate"].T) * ple[:, i]) @ w["per_layer_proj"].T
        x = x + unit(y, EPS) * w["per_layer_post_norm"]
    if not lanes:
        x = x[-1:]
    y = unit(x, EPS) * m["output_norm"].to(F64)
    z = torch.cat([y @ unpack(m["embed"][lo:lo + 16384]).T for lo in range(0, c["vocab"], 16384)], 1)
    z = 30.0 * torch.tanh(z / 30.0)
    return z if lanes else z.cpu().numpy()


def decoder_work(c):
    cfg, R, T = decoder_config(c), c["rows"], c["context"]
    packed = {"q4_0": 18 / 32, "tq2_0": 66 / 256}
    nbytes, values, scores = 0.0, 0.0, 0.0
    for i in range(c["layers"]):
        for fmt, n, k in decoder_shapes(c, cfg, i).values():
            nbytes, values = nbytes + n * k * packed[fmt], values + n * k
        hd, seen = cfg.attn_head_dim(i), T if cfg.is_full_attention(i) else min(T, WINDOW)
        mean = 0.75 * seen if c["mode"] == "lanes" and cfg.is_full_attention(i) else seen
        nbytes += mean * (hd // 2 + 4) * (R if c["mode"] == "lanes" else 1)
        scores += 4 * R * HEADS * hd * mean
    out_rows = R if c["mode"] == "lanes" else 1
    head = c["vocab"] * c["hidden"]
    proj = c["layers"] * PER_LAYER * c["hidden"]
    return {"bytes": nbytes + (head + proj) * packed["q4_0"] + out_rows * c["vocab"] * 4, "flops": 2 * R * (values + proj) + 2 * out_rows * head + scores}


# ---- stacks with bf16 weights -------------------------------------------------------------------------------------------
def stack_config(c):
    """Four layers, as config.json has them: every kind of token mixer of the design, dense and routed feed-forwards."""
    w = c["width"]
    H = w // 128

    def layer(kind, mixer, ff):
        return {"type": kind, "mixer": mixer, "mlp": ff}
    if c["design"] == "Komirax":
        kv = max(k for k in (1, 2, 3, 4) if H % k == 0)
        attn = {"heads": H, "kv_heads": kv, "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.3}
        lin = {"heads": H, "dim": 128, "vdim": 128, "decay": list(np.linspace(0.9, 0.999, H))}
        dense = {"kind": "dense", "ff": 4 * w}
        moe = {"kind": "moe", "router": {"experts": H, "top": 2}, "expert": {"ff": w // 2}}
        layers = [layer("attention", attn, dense), layer("lightning", lin, dense), layer("attention", attn, moe), layer("lightning", lin, moe)]
        return {"architecture": "Komirax", "vocab": c["vocab"], "width": w, "norm": {"eps": 1e-6}, "layers": layers, "loop": None}
    lat = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5}
    ret = {"heads": H, "dim": 128, "vdim": 128, "decay": list(1.0 - 2.0 ** -np.linspace(3, 9, H))}
    ssm = {"heads": w // 32, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    ff = {"kind": "dense", "ff": w * 8 // 3 // 64 * 64}
    layers = [layer("latent_attention", lat, ff), layer("latent_attention", {**lat, "kv_from": 0}, ff), layer("retention", ret, ff), layer("mamba2", ssm, ff)]
    return {"architecture": "Vifivik", "vocab": c["vocab"], "width": w, "norm": {"eps": 1e-6}, "layers": layers, "logit_softcap": 30.0}


class Weights:
    """A model's weights as the loader asks for them: names to bf16 values on the device."""

    def __init__(self, cfg, src):
        self.t, w, v, deep = {}, cfg["width"], cfg["vocab"], cfg["architecture"] == "Komirax"

        def put(name, x):
            self.t[name] = x.bfloat16()

        def mat(name, rows, cols, scale=1.0):
            put(name, src.normal(rows, cols) * (scale / math.sqrt(cols)))

        def norm(name, n, mean=1.0):
            put(name, mean + 0.1 * src.normal(n))
        experts = max([l["mlp"]["router"]["experts"] for l in cfg["layers"] if l["mlp"]["kind"] == "moe"] or [0])
        embed = src.normal(v, w) * (0.5 if deep else 1.0)
        if experts:                                        # tokens have favourite experts, as after training
            dirs = torch.linalg.qr(src.normal(w, w))[0][:experts]
            embed -= embed @ dirs.T @ dirs
            embed += (src.order(experts, v) - (experts - 1) / 2) * (2 * math.sqrt(w) / experts) @ dirs
        put("embed", embed)
        for i, l in enumerate(cfg["layers"]):
            p, m, f = f"l{i}.mix.", l["mixer"], l["mlp"]
            H, e = m["heads"], m["vdim"]
            norm(f"l{i}.norm1", w, 1.0 if deep else 0.5)
            if l["type"] == "attention":
                for n, k in (("q", H * 2 * m["dim"]), ("k", m["kv_heads"] * 2 * m["dim"]), ("v", m["kv_heads"] * e)):
                    mat(p + n, k, w)
                    put(f"{p}{n}.b", 0.3 * src.normal(k))
                for n in ("lq1", "lk1", "lq2", "lk2"):
                    put(p + n, 0.8 / math.sqrt(m["dim"]) * src.normal(m["dim"]))
                mat(p + "o", w, H * e, 0.4)
            elif l["type"] in ("lightning", "retention"):
                for n, k in (("q", H * m["dim"]), ("k", H * m["dim"]), ("v", H * e), ("g", H * e)):
                    mat(p + n, k, w)
                mat(p + "o", w, H * e, 0.4 if deep else 1.0)
                if deep:
                    norm(p + "norm", H * e)
            elif l["type"] == "latent_attention":
                d, z, r = m["dim"], m["rot_dim"], m["kv_rank"]
                mat(p + "q", H * (d + z), w, 1.5)
                if "kv_from" not in m:
                    mat(p + "dkv", r + z, w)
                    norm(p + "dkv.norm", r)
                mat(p + "uk", H * d, r)
                mat(p + "uv", H * e, r)
                put(p + "sink", 1.5 * src.normal(H))
                mat(p + "g", H, w)
                mat(p + "o", w, H * e)
            else:
                inner, ch = H * e, H * e + 2 * m["groups"] * m["state"]
                mat(p + "in", inner + ch + H, w)
                mat(p + "conv", ch, m["conv"], 1.5)
                put(p + "conv.b", 0.2 * src.normal(ch))
                put(p + "dt_bias", torch.linspace(-5.0, -0.5, H, device=DEVICE))
                put(p + "A_log", torch.linspace(2.0, -1.0, H, device=DEVICE))
                put(p + "D", src.normal(H))
                norm(p + "norm", inner)
                mat(p + "o", w, inner)
            p = f"l{i}.mlp."
            norm(f"l{i}.norm2", w, 1.0 if deep else 0.5)
            if f["kind"] == "moe":
                put(p + "router", dirs[src.order(experts, 1)[0]] * 1.5)
                for j in range(experts):
                    mat(f"{p}e{j}.up", f["expert"]["ff"], w)
                    mat(f"{p}e{j}.down", w, f["expert"]["ff"], 0.3)
            else:
                for n in ("up",) if deep else ("gate", "up"):
                    mat(p + n, f["ff"], w)
                mat(p + "down", w, f["ff"], 0.6 if deep else 1.0)
        norm("final.norm", w)
        mat("head", v, w, 2.0 if deep else 4.0)

    def bf16(self, name, shape=None):
        x = self.t[name]
        assert shape is None or x.shape == tuple(shape), name
        return x.view(torch.int16).cpu().numpy().view(np.uint16)

    def f32(self, name, shape=None):
        assert shape is None or self.t[name].shape == tuple(shape), name
        return self.t[name].float().cpu().numpy()

    def __getitem__(self, name):
        return self.t[name].to(F64)


def stack_inputs(c, seed):
    src = Source(seed)
    cfg = stack_config(c)
    return cfg, Weights(cfg, src), src.whole(c["vocab"], c["prompt"] + c["new"]).tolist()


def stack_prepare(c, seed):
    ctx, K = context()
    cfg, weights, tokens = stack_inputs(c, seed)
    dtype = TYPE[c["dtype"]][0]
    model = pkg.stack_pipeline.StackPipeline(ctx, K, pkg.registry.read_config(cfg), weights, c["prompt"] + c["new"], dtype)
    return {"case": c, "model": model, "tokens": tokens}


def stack_run(s):
    c, model, tokens = s["case"], s["model"], s["tokens"]
    seq, P, logits = model.new_sequence(), c["prompt"], []
    for lo in range(0, P, c["portion"]):
        hi = min(lo + c["portion"], P)
        got = model.step(seq, tokens[lo:hi], [hi - lo - 1] if hi == P else [])
    logits.append(got)
    for t in tokens[P:]:
        logits.append(model.step(seq, [t], [0]))
    model.end_sequence(seq)
    return np.concatenate(logits)


def silu(x):
    return x * torch.sigmoid(x)


def decayed(q, k, v, steps):
    """One head's causal linear attention: k's row j reaches q's row i through exp(steps[i] - steps[j])."""
    d = steps[:, None] - steps[None]
    return (q @ k.T * torch.exp(d.masked_fill(d.new_ones(d.shape, dtype=torch.bool).triu(1), -math.inf))) @ v


def causal(q, k, v, scale, sink=None):
    z = (q @ k.T * scale).masked_fill(torch.ones(len(q), len(q), device=DEVICE, dtype=torch.bool).triu(1), -math.inf)
    if sink is not None:
        z = torch.cat([z, sink.expand(len(q), 1)], 1)
    return torch.softmax(z, 1)[:, :len(q)] @ v


def mixed(l, w, p, h, eps, cache):
    """The token mixer of one layer over a whole sequence, float64 [T, width]."""
    m, T = l["mixer"], h.shape[0]
    H, e, kind = m["heads"], m["vdim"], l["type"]
    if kind == "attention":
        d, kv = m["dim"], m["kv_heads"]
        q, k, v = (h @ w[p + n].T + w[f"{p}{n}.b"] for n in "qkv")
        q, k, v = q.reshape(T, H, 2, d), k.reshape(T, kv, 2, d), v.reshape(T, kv, e)
        lam = torch.exp((w[p + "lq1"] * w[p + "lk1"]).sum()) - torch.exp((w[p + "lq2"] * w[p + "lk2"]).sum()) + m["diff"]
        o = [[causal(q[:, i, j], k[:, i * kv // H, j], v[:, i * kv // H], m["scale"]) for j in (0, 1)] for i in range(H)]
        o = torch.stack([unit(a - lam * b, eps) * (1 - m["diff"]) for a, b in o], 1)
    elif kind in ("lightning", "retention"):
        act = silu if kind == "lightning" else (lambda x: x)
        q, k, v = (act(h @ w[p + n].T).reshape(T, H, -1) for n in "qkv")
        k = k if kind == "lightning" else k * m["dim"] ** -0.5
        steps = torch.arange(T, device=DEVICE, dtype=F64)
        # the decays as the model holds them: 32-bit
        o = torch.stack([decayed(q[:, i], k[:, i], v[:, i], steps * math.log(np.float32(m["decay"][i]))) for i in range(H)], 1)
        g = h @ w[p + "g"].T
        o = unit(o.reshape(T, -1), eps) * w[p + "norm"] * torch.sigmoid(g) if kind == "lightning" else unit(o, eps).reshape(T, -1) * silu(g)
    elif kind == "latent_attention":
        d, z, r = m["dim"], m["rot_dim"], m["kv_rank"]
        a = torch.arange(T, device=DEVICE, dtype=F64)[:, None] * m["rot"]["base"] ** (-2.0 * torch.arange(z // 2, device=DEVICE, dtype=F64) / z)

        def turn(x):                                       # [T, heads, z]: neighbours are pairs
            u, v = x[..., 0::2], x[..., 1::2]
            return torch.stack([u * a.cos()[:, None] - v * a.sin()[:, None], v * a.cos()[:, None] + u * a.sin()[:, None]], 3).flatten(2)
        if "kv_from" not in m:
            x = h @ w[p + "dkv"].T
            cache["latent"], cache["rotated"] = unit(x[:, :r], eps) * w[p + "dkv.norm"], turn(x[:, None, r:])[:, 0]
        q = (h @ w[p + "q"].T).reshape(T, H, d + z)
        q = torch.cat([q[..., :d], turn(q[..., d:])], 2)
        k, v = (cache["latent"] @ w[p + "uk"].T).reshape(T, H, d), (cache["latent"] @ w[p + "uv"].T).reshape(T, H, e)
        gate = torch.sigmoid(h @ w[p + "g"].T)
        o = torch.stack([gate[:, i:i + 1] * causal(q[:, i], torch.cat([k[:, i], cache["rotated"]], 1), v[:, i], m["scale"], w[p + "sink"][i]) for i in range(H)], 1)
    else:
        inner, n = H * e, m["groups"] * m["state"]
        x = h @ w[p + "in"].T
        z, u, dt = x[:, :inner], x[:, inner:2 * inner + 2 * n], x[:, 2 * inner + 2 * n:]
        taps, u = w[p + "conv"], torch.cat([u.new_zeros(m["conv"] - 1, u.shape[1]), u])
        u = silu(w[p + "conv.b"] + sum(u[j:j + T] * taps[:, j] for j in range(m["conv"])))
        x, B, C = u[:, :inner].reshape(T, H, e), u[:, inner:inner + n].reshape(T, m["groups"], -1), u[:, inner + n:].reshape(T, m["groups"], -1)
        dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"])
        steps = torch.cumsum(-torch.exp(w[p + "A_log"]) * dt, 0)
        per = H // m["groups"]
        o = [decayed(C[:, i // per], B[:, i // per] * dt[:, i:i + 1], x[:, i], steps[:, i]) + w[p + "D"][i] * x[:, i] for i in range(H)]
        o = torch.stack(o, 1).reshape(T, inner) * silu(z)
        o = unit(o.reshape(T, m["norm_groups"], -1), eps).reshape(T, inner) * w[p + "norm"]
    return o.reshape(T, -1) @ w[p + "o"].T


def fed_forward(f, w, p, h, before):
    if f["kind"] == "moe":
        z = h @ w[p + "router"].T
        best = z.topk(f["router"]["top"], 1).indices
        y = torch.zeros_like(h)
        for j in range(f["router"]["experts"]):
            at = (best == j).any(1).nonzero()[:, 0]
            x = torch.relu((torch.sigmoid(z[at, j:j + 1]) * h[at]) @ w[f"{p}e{j}.up"].T) ** 2
            y[at] += x @ w[f"{p}e{j}.down"].T
        return y
    if before:
        return gelu_tanh(h @ w[p + "up"].T) @ w[p + "down"].T
    return (silu(h @ w[p + "gate"].T) * (h @ w[p + "up"].T)) @ w[p + "down"].T


def stack_exact(c, seed):
    cfg, w, tokens = stack_inputs(c, seed)
    eps, before, cache = cfg["norm"]["eps"], cfg["architecture"] == "Komirax", {}
    x = w["embed"][torch.tensor(tokens, device=DEVICE)]
    for i, l in enumerate(cfg["layers"]):
        for name, branch in (("norm1", lambda h: mixed(l, w, f"l{i}.mix.", h, eps, cache)), ("norm2", lambda h: fed_forward(l["mlp"], w, f"l{i}.mlp.", h, before))):
            n = w[f"l{i}.{name}"]
            x = x + (branch(unit(x, eps) * n) if before else unit(branch(x), eps) * n)
    z = (unit(x[c["prompt"] - 1:], eps) * w["final.norm"]) @ w["head"].T
    cap = cfg.get("logit_softcap")
    return (cap * torch.tanh(z / cap) if cap else z).cpu().numpy()


def stack_work(c):
    cfg, w, P, N = stack_config(c), c["width"], c["prompt"], c["new"]
    passes, L = -(-P // min(c["portion"], 2048)) + N, P + N
    always = chosen = experts = 0                           # weights every token meets; of one token's experts; of all experts
    pair = state = 0.0                                      # flops per visible pair of tokens; per token in recurrences
    cached = 0                                              # bytes a token leaves in caches
    for l in cfg["layers"]:
        m, f = l["mixer"], l["mlp"]
        H, e = m["heads"], m["vdim"]
        if l["type"] == "attention":
            always += w * (2 * m["dim"] * (H + m["kv_heads"]) + e * (H + m["kv_heads"]))
            pair += 4 * H * (m["dim"] + e)
            cached += m["kv_heads"] * (2 * m["dim"] + e) * 2
        elif l["type"] in ("lightning", "retention"):
            always += w * H * (2 * m["dim"] + 3 * e)
            state += 4 * H * m["dim"] * e
        elif l["type"] == "latent_attention":
            own = "kv_from" not in m
            always += w * (H * (m["dim"] + m["rot_dim"] + 1 + e) + (m["kv_rank"] + m["rot_dim"]) * own) + H * (m["dim"] + e) * m["kv_rank"]
            pair += 2 * H * (m["dim"] + m["rot_dim"] + e)
            cached += (m["kv_rank"] + m["rot_dim"]) * 2 * own
        else:
            always += w * (3 * H * e + 2 * m["groups"] * m["state"] + H)
            state += 4 * H * m["state"] * e
        if f["kind"] == "moe":
            each = 2 * w * f["expert"]["ff"]
            always, chosen, experts = always + w * f["router"]["experts"], chosen + each * f["router"]["top"], experts + each * f["router"]["experts"]
        else:
            always += w * f["ff"] * (2 if cfg["architecture"] == "Komirax" else 3)
    head = w * c["vocab"]
    nbytes = 2 * (passes * always + (passes - N) * experts + N * chosen + (N + 1) * head) + cached * (L + N * (P + N / 2)) + (N + 1) * c["vocab"] * 4 + L * w * 2
    return {"bytes": nbytes, "flops": L * (2 * (always + chosen) + state) + pair * L * L / 2 + 2 * (N + 1) * head}


# ---- single dispatches --------------------------------------------------------------------------------------------------
def matvec_inputs(c, seed):
    src = Source(seed)
    return [src.blocks(c["format"], c["rows"], c["cols"]) for _ in range(c["count"])], src.normal(c["count"], c["cols"])


def matvec_prepare(c, seed):
    raw, x = matvec_inputs(c, seed)
    y = torch.empty(c["count"], c["rows"], device=DEVICE)
    return {"case": c, "w": [upload(r) for r in raw], "x": [wrap(v) for v in x], "y": y, "out": [wrap(v) for v in y], "batch": pkg.CommandBatch(context()[0])}


def matvec_run(s):
    c = s["case"]
    context()[1].matvec_quant_grouped_into(s["batch"], FORMAT[c["format"]], s["w"], s["x"], pkg.F32, s["out"], pkg.F32, c["rows"], c["cols"])
    return s["y"]


def matvec_exact(c, seed):
    raw, x = matvec_inputs(c, seed)
    return torch.stack([unpack(r) @ v.to(F64) for r, v in zip(raw, x)])


def matvec_work(c):
    n, k = c["rows"], c["cols"]
    return {"bytes": c["count"] * (n * k * (18 / 32 if c["format"] == "q4_0" else 66 / 256) + 4 * (n + k)), "flops": 2.0 * c["count"] * n * k}


def matmul_inputs(c, seed):
    src = Source(seed)
    return src.blocks(c["format"], c["n"], c["k"]), src.normal(c["m"], c["k"]).to(TYPE[c["input"]][1])


def matmul_prepare(c, seed):
    raw, x = matmul_inputs(c, seed)
    w = pkg.QuantWeight.quantized(upload(raw), FORMAT[c["format"]], c["n"], c["k"])
    y = torch.empty(c["m"], c["n"], device=DEVICE, dtype=TYPE[c["output"]][1])
    return {"case": c, "w": w, "x": wrap(x), "y": y, "out": wrap(y), "batch": pkg.CommandBatch(context()[0])}


def matmul_run(s):
    c = s["case"]
    s["w"].matmul_nt_typed_into(s["batch"], context()[1], s["x"], TYPE[c["input"]][0], s["out"], TYPE[c["output"]][0], c["m"])
    return s["y"]


def matmul_exact(c, seed):
    raw, x = matmul_inputs(c, seed)
    return x.to(F64) @ unpack(raw).T


def matmul_work(c):
    m, k, n = c["m"], c["k"], c["n"]
    size = {"bf16": 2, "f16": 2, "f32": 4}
    return {"bytes": n * k * (18 / 32 if c["format"] == "q4_0" else 66 / 256) + m * k * size[c["input"]] + m * n * size[c["output"]], "flops": 2.0 * m * k * n}


def attention_prepare(c, seed):
    """A pool of sequences of one length; a sliding window reads the end of each."""
    ctx, K = context()
    src, hd, T, lanes = Source(seed), c["head_dim"], c["context"], c["lanes"]
    pool = pkg.QuantizedUnifiedKvPool(ctx, lanes, T, 1, hd, 2)
    for codes, norms in ((pool.keys_q, pool.key_norms), (pool.values_q, pool.value_norms)):
        for lo in range(0, lanes * T, 1 << 19):
            n = min(lanes * T - lo, 1 << 19)
            rows = src.normal(n, hd).half()
            torch.cuda.synchronize()
            batch = pkg.CommandBatch(ctx)
            K.encode_kv_turboquant_into(batch, wrap(rows), pool.levels, pool.signs, codes, norms, hd, 1, n, 2, lo, 0)
            batch.commit_and_wait()
    q = src.normal(lanes, HEADS, hd) * hd ** -0.5                 # rotated queries; keys of N(0, 1): scores of about unit spread
    positions = torch.full((lanes,), T - 1, device=DEVICE, dtype=torch.int32)
    out = torch.empty(lanes, HEADS, hd, device=DEVICE)
    return {"case": c, "pool": pool, "q": q, "out": out, "positions": positions, "buffers": [wrap(t) for t in (q, out, positions)], "batch": pkg.CommandBatch(ctx)}


def attention_run(s):
    c, p = s["case"], s["pool"]
    q, out, positions = s["buffers"]
    context()[1].flash_attention_tq_batched_into(s["batch"], q, p.keys_q, p.key_norms, p.values_q, p.value_norms, p.levels, out, positions, c["head_dim"],
                                                 p.lane_stride(), HEADS, 1, c["window"], 2, c["lanes"], 0)
    return s["out"]


def attention_exact(c, seed):
    s = attention_prepare(c, seed)
    p, T, hd = s["pool"], c["context"], c["head_dim"]
    levels, first = on_device(p.levels.as_array(np.float32)).to(F64), max(0, T - c["window"]) if c["window"] else 0
    k, v = on_device(p.keys_q.as_array(np.uint8)), on_device(p.values_q.as_array(np.uint8))
    kn, vn = (on_device(b.as_array(np.float16)).to(F64) for b in (p.key_norms, p.value_norms))

    def rows(codes, norms, lane):
        b = codes[lane * T * hd // 4:(lane + 1) * T * hd // 4].reshape(T, hd // 4, 1)[first:]
        return levels[torch.cat([b >> 2 * i & 3 for i in range(4)], 2).reshape(T - first, hd).long()] * norms[lane * T + first:(lane + 1) * T, None]
    return torch.stack([torch.softmax(s["q"][i].to(F64) @ rows(k, kn, i).T, 1) @ rows(v, vn, i) for i in range(c["lanes"])])


def attention_work(c):
    seen, hd = min(c["context"], c["window"] or c["context"]), c["head_dim"]
    return {"bytes": c["lanes"] * (seen * (hd // 2 + 4) + 8 * HEADS * hd), "flops": 4.0 * c["lanes"] * HEADS * hd * seen}


# ---- what is called from outside ----------------------------------------------------------------------------------------
KINDS = {"decoder": (decoder_prepare, decoder_run, decoder_exact, decoder_work), "stack": (stack_prepare, stack_run, stack_exact, stack_work),
         "matvec": (matvec_prepare, matvec_run, matvec_exact, matvec_work), "matmul": (matmul_prepare, matmul_run, matmul_exact, matmul_work),
         "attention": (attention_prepare, attention_run, attention_exact, attention_work)}


def prepare(case, seed):
    s = KINDS[case["kind"]][0](case, seed)
    torch.cuda.synchronize()
    return s


def run(state):
    return KINDS[state["case"]["kind"]][1](state)


def work(case):
    return KINDS[case["kind"]][3](case)


def exact(case, seed):
    return KINDS[case["kind"]][2](case, seed)


def tolerance(case):
    """About four times what the framework and the 64-bit statement differ by."""
    if case["kind"] == "decoder":                           # f16 between kernels; 2-bit codes of new rows fall either way
        return {"rel": 0.02, "max": 0.3}
    if case["kind"] == "stack":
        return {"rel": 0.02, "max": 0.3} if case["dtype"] == "bf16" else {"rel": 1e-5, "max": 2e-4}
    return {"rel": 1e-3, "max": 1e-2}
