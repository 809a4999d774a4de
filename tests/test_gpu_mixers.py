"""The kernels for models with bf16 weights, each against plain f64 arithmetic: products by segments in every form, norms,
softmax attention with one and two maps over block caches, linear attention (recurrent and chunked), mixture of experts."""
import numpy as np
import pytest

import mixer_models as M
from oracle import mixer_stack as O

pytestmark = pytest.mark.gpu

F32_TOL, BF16_TOL = 2e-5, 1.2e-2      # of the largest wanted value


@pytest.fixture(scope="module")
def ai(pkg):
    import local_ai_amd
    return local_ai_amd


def upload(ai, ctx, x, dtype):
    return ai.Buffer.from_slice(ctx, M.bf16_bits(x) if dtype == ai.BF16 else np.asarray(x, np.float32))


def download(ai, buf, count, dtype):
    return M.bf16_values(buf.as_array(np.uint16, count)) if dtype == ai.BF16 else buf.as_array(np.float32, count)


def empty(ai, ctx, count, dtype):
    return ai.Buffer.empty(ctx, count * (2 if dtype == ai.BF16 else 4))


def stored(x, ai, dtype):
    return M.rounded(x) if dtype == ai.BF16 else np.asarray(x, np.float32).astype(np.float64)


def close(got, want, tol, what=""):
    err = np.abs(got - want).max() / max(np.abs(want).max(), 1e-9)
    assert np.isfinite(got).all() and err <= tol, f"{what}: {err:.3g}"


ACTS = [lambda z: z, O.silu, O.gelu_tanh, O.relu_squared, O.sigmoid]


def block_order():
    """Place of each of a value block's 32 positions."""
    return np.array([((p >> 2) & 3) * 8 + ((p >> 4) & 1) * 4 + (p & 3) for p in range(32)])


def values_from_cache(flat, cols):
    """[positions, cols] from [block][cols][32]."""
    b = flat.reshape(-1, cols, 32)[:, :, block_order()]
    return b.transpose(0, 2, 1).reshape(-1, cols)


# ---- products ----------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("cols,shift", [(1, 0), (4, 0), (7, 0), (1023, 0), (1024, 0), (1028, 0), (2048, 1), (5000, 0)])
def test_embed_token(ai, gpu, cols, shift):
    ctx, K = gpu
    table = M.rounded(np.random.default_rng(cols).standard_normal((5, cols)))
    tb = ai.Buffer.from_slice(ctx, np.concatenate([np.zeros(shift, np.uint16), M.bf16_bits(table).reshape(-1)])).view(2 * shift, 10 * cols)
    out, at, then, batch = ai.Buffer.from_slice(ctx, np.full(cols + 4, 7, np.float32)), ai.Buffer.empty(ctx, 4), ai.Buffer.empty(ctx, 4), ai.CommandBatch(ctx)
    for token in (3, 0, 4, 9):
        K.embed_token_bf16_into(batch, tb, 5, cols, token, 40 + token, out, at, then)
        batch.commit_and_wait()
        got = out.as_array(np.float32, cols + 4)
        assert np.array_equal(got[:cols], table[min(token, 4)]) and (got[cols:] == 7).all()
        assert at.as_array(np.uint32, 1)[0] == 40 + token and then.as_array(np.uint32, 1)[0] == 41 + token


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("m,k,n", [(1, 64, 48), (2, 256, 200), (31, 72, 33), (33, 40, 70), (64, 520, 130), (65, 64, 64), (129, 200, 257),
                                   (300, 136, 2052), (7, 60, 45), (140, 7, 9), (2100, 128, 2048),
                                   (1, 4104, 300), (1, 5000, 17), (1, 8192, 70), (1, 16384, 9), (1, 20008, 5), (1, 16, 270000), (600, 2048, 1100)])
def test_linear_rows(ai, gpu, dtype, m, k, n):
    ctx, K = gpu
    dt = ai.BF16 if dtype == "bf16" else ai.F32
    g = np.random.default_rng(m + k + n)
    x, w, b = stored(g.standard_normal((m, k)), ai, dt), M.rounded(g.standard_normal((n, k)) / np.sqrt(k)), g.standard_normal(n).astype(np.float32)
    want = x @ w.T + b
    print(f"linear {dtype} {m} {k} {n}", flush=True)
    xb, L = upload(ai, ctx, x, dt), ai.linear_weight
    act = (m + n) % 5
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(n, act)], [b])
    out, res = empty(ai, ctx, m * n, ai.F32), upload(ai, ctx, np.ones((m, n)), ai.F32)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, xb, dt, m, [out], ai.F32)
    lin.rows_add_into(batch, K, xb, dt, m, res)
    batch.commit_and_wait()
    close(download(ai, out, m * n, ai.F32).reshape(m, n), ACTS[act](want), F32_TOL, "f32 output")
    close(download(ai, res, m * n, ai.F32).reshape(m, n), ACTS[act](want) + 1, F32_TOL, "residual")
    if m == 1:
        v = empty(ai, ctx, n, ai.F32)
        K.linear_vector_into(batch, xb, dt, lin.weight, lin.bias, k, lin.segments, [v], ai.F32)
        batch.commit_and_wait()
        close(download(ai, v, n, ai.F32), ACTS[act](want)[0], F32_TOL, "vector")


@pytest.mark.parametrize("m,k,n", [(2048, 64, 8192), (1990, 192, 8176), (1793, 128, 8150), (2048, 320, 3072), (1830, 64, 2064), (1500, 256, 3000), (2048, 192, 2048),
                                   (1930, 64, 2000), (1921, 448, 1936), (2048, 576, 1920)])
@pytest.mark.parametrize("act", [0, 1, 2, 3])
def test_large_products(ai, gpu, m, k, n, act):
    """The 256 x 256, 256 x 128 and 128 x 128 tiles of large products: whole and ragged, one step of k to nine, every way a lane
    finishes its columns; bf16 and f32 outputs, with and without the residual."""
    ctx, K = gpu
    g = np.random.default_rng(m + k + n)
    x, w, b = M.rounded(g.standard_normal((m, k))), M.rounded(g.standard_normal((n, k)) / np.sqrt(k)), g.standard_normal(n).astype(np.float32)
    want = ACTS[act](x @ w.T + b)
    L = ai.linear_weight
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(n, act)], [b])
    xb, out, wide, res = upload(ai, ctx, x, ai.BF16), empty(ai, ctx, m * n, ai.BF16), empty(ai, ctx, m * n, ai.F32), upload(ai, ctx, np.ones((m, n)), ai.F32)
    print(f"large product {m} {k} {n} {act}", flush=True)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, xb, ai.BF16, m, [out], ai.BF16)
    lin.rows_into(batch, K, xb, ai.BF16, m, [wide], ai.F32)
    lin.rows_add_into(batch, K, xb, ai.BF16, m, res)
    batch.commit_and_wait()
    got = download(ai, out, m * n, ai.BF16).reshape(m, n)
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + F32_TOL * np.abs(want).max()).all()      # one rounding to bf16
    close(download(ai, wide, m * n, ai.F32).reshape(m, n), want, F32_TOL, "f32 output")
    close(download(ai, res, m * n, ai.F32).reshape(m, n), want + 1, F32_TOL, "residual")


@pytest.mark.parametrize("m,k,n", [(33, 8, 36), (64, 576, 512), (100, 4096, 260), (129, 200, 1000), (511, 1288, 1028), (512, 2048, 1024), (480, 712, 1536),
                                   (33, 72, 36), (33, 136, 36), (301, 1048, 712), (333, 1000, 1032), (190, 4104, 1500), (333, 2056, 1036), (287, 176, 1444), (2100, 2056, 2080), (1500, 712, 1512), (1490, 1096, 2308)])
@pytest.mark.parametrize("act", [0, 1, 2, 3])
def test_products_of_few_tiles(ai, gpu, m, k, n, act):
    """By the rule for 256 CUs.  Waves that share out k on 32 x 32 tiles: 64 x 512 x 576, 100 x 260 x 4096, 129 x 1000 x 200, 301 x 712 x 1048
    and, with f32 results, 33 rows of k 72 and 136, which leave waves without a step; on 64 x 32: 512 x 1024 x 2048 and, with ragged rows,
    columns and last steps, those of k 1000, 4104 and 2056 and f32 results of k 1288.  Shared waves: 32 x 32 for k 8 and 176 and bf16 results of k 72
    and 136; 64 x 64 with four buffers for 480 rows of k 712 and bf16 results of k 1288, with three for 1500 rows; 128 x 64 for
    1490 rows and 128 x 128 for 2100."""
    test_large_products(ai, gpu, m, k, n, act)


@pytest.mark.parametrize("act", ["silu", "gelu", "pairs"])
@pytest.mark.parametrize("m", [1024, 64])
def test_activations_of_bf16_results(ai, gpu, act, m):
    """Activations of many rows round to bf16 from 32-bit values, infinities and NaN as f32 arithmetic has them.  A result lies half a
    bf16 step from the f64 activation of the same f32 sum, and 7 x 2^-24 of its size: the exponential (one ulp, two of these units), the
    constant ln 2 (one, up to |z| = 20), two sums and the quotient (one each), a second factor (one); gelu's argument carries three roundings,
    which the exponential multiplies by its size."""
    ctx, K = gpu
    g, L, n, k = np.random.default_rng(m), ai.linear_weight, 4096, 64
    x, w, b = M.rounded(g.uniform(-4, 4, m)), M.rounded(g.uniform(-4, 4, n)), g.uniform(-4, 4, n).astype(np.float32)
    b[:16] = (np.inf, -np.inf, np.nan, 3e38, -3e38, 88.5, -88.5, -86.0, -95.0, 130.0, -130.0, 0.0, -0.0, 1e-30, -1e-30, -1e20)
    w[:16] = 0.0
    xs, ws = np.zeros((m, k)), np.zeros((n, k))
    xs[:, 0], ws[:, 0] = x, w                               # one exact product and one addition: the sum is known to the bit
    lin = L.StackedLinear(ctx, [M.bf16_bits(ws)], [L.Segment(n, {"silu": ai.ACT_SILU, "gelu": ai.ACT_GELU_TANH, "pairs": ai.ACT_SILU_PAIRS}[act])], [b])
    width = n // 2 if act == "pairs" else n
    out, batch = empty(ai, ctx, m * width, ai.BF16), ai.CommandBatch(ctx)
    print(f"activations {act} {m}", flush=True)
    lin.rows_into(batch, K, upload(ai, ctx, xs, ai.BF16), ai.BF16, m, [out], ai.BF16)
    batch.commit_and_wait()
    got = download(ai, out, m * width, ai.BF16).reshape(m, width)
    v = ((x[:, None] * w).astype(np.float32) + b).astype(np.float64)
    with np.errstate(all="ignore"):
        first, second = (v[:, 0::2], v[:, 1::2]) if act == "pairs" else (v, 1.0)
        z = 1.5957691216057308 * (first + 0.044715 * first ** 3) if act == "gelu" else first
        e = np.exp(-z)
        want = first / (1.0 + e) * second
        slack = (7 + 3 * np.minimum(np.abs(z), 100) * e / (1 + e) * (act == "gelu")) * 2.0 ** -24
        half = np.exp2(np.floor(np.log2(np.abs(want)))) * 2.0 ** -8
        usual = np.isfinite(v[:, 0::2] + v[:, 1::2] if act == "pairs" else v) & (np.abs(z) < 20) & (np.abs(want) > 1e-30) & (np.abs(want) < 3e38)
        assert usual.mean() > 0.6
        over = (np.abs(got - want) - half) / np.abs(want) / 2.0 ** -24
        assert (over <= slack * 2.0 ** 24)[usual].all(), over[usual].max()
        plain = empty(ai, ctx, m * width, ai.F32)              # f32 results go through expf and a division
        lin.rows_into(batch, K, upload(ai, ctx, xs, ai.BF16), ai.BF16, m, [plain], ai.F32)
        batch.commit_and_wait()
        missed, expected = (int((np.abs(r - want) > half)[usual].sum()) for r in (got, M.rounded(download(ai, plain, m * width, ai.F32).reshape(m, width))))
        print(f"not nearest: {missed}, rounded from f32 {expected}, of {usual.sum()}", flush=True)
        assert missed <= 1.2 * expected + 8
        alone = ai.Buffer.empty(ctx, 4 * width)               # a single row keeps expf and the division
        lin.vector_into(batch, K, upload(ai, ctx, xs[0], ai.F32), ai.F32, [alone], ai.F32)
        batch.commit_and_wait()
        special, same = got[0, :16 if width == n else 8], M.rounded(alone.as_array(np.float32, width)[:16 if width == n else 8])
        assert np.array_equal(np.isnan(special), np.isnan(same)) and np.allclose(special, same, 2.0 ** -7, 1e-36, equal_nan=True), (special, same)


@pytest.mark.parametrize("m,k,n", [(40, 72, 50), (333, 1024, 256), (2048, 64, 2048), (3, 4096, 16)])
def test_f32_rows_as_terms(ai, gpu, m, k, n):
    """32-bit activations on the matrix cores: all 24 bits of every value, whatever its size, and what is infinite or no number comes
    out as f32 products and sums have it."""
    ctx, K = gpu
    g, L = np.random.default_rng(m + k), ai.linear_weight
    x, w = (g.standard_normal((m, k)) * 10.0 ** g.integers(-6, 7, (m, k))).astype(np.float32), M.rounded(g.standard_normal((n, k)) / np.sqrt(k))
    x[0, 5], x[1, 0], x[2, 1:3] = np.inf, np.nan, (np.inf, -np.inf)
    w[1, 5], w[2, 7], w[3, 5] = np.inf, -np.inf, 0.0
    w[4, 3:5] = np.inf, np.nan
    x[:, 7] = np.where(np.arange(m) % 3 == 0, 0.0, np.where(np.arange(m) % 3 == 1, 1.5, -2.0 ** -20))
    xd = x.astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = np.stack([(xd * r).sum(1) for r in w], 1)
        size = np.abs(np.where(np.isfinite(xd), xd, 0.0)) @ np.abs(np.where(np.isfinite(w), w, 0.0)).T
    out = empty(ai, ctx, m * n, ai.F32)
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(n)])
    print(f"terms {m} {k} {n}", flush=True)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, upload(ai, ctx, x, ai.F32), ai.F32, m, [out], ai.F32)
    batch.commit_and_wait()
    got = download(ai, out, m * n, ai.F32).reshape(m, n)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    # a rounding for each 32 exact products of each of the three terms, and the product's own 32
    assert (np.abs(got[fine] - want[fine]) <= ((3 * k / 32 + 32) * 2.0 ** -24 * size)[fine]).all()


@pytest.mark.parametrize("m,k,n", [(1536, 1024, 32), (1537, 1024, 32), (1001, 2120, 40)])
def test_f32_rows_as_terms_around_the_line(ai, gpu, m, k, n):
    """Around the workgroups beyond which a lane makes four trips, and with rows that end within one."""
    test_f32_rows_as_terms(ai, gpu, m, k, n)


@pytest.mark.parametrize("bits", [1, 2, 7, 8, 9, 15, 16, 17, 24])
def test_terms_of_small_f32_values(ai, gpu, bits):
    """Values of every number of bits from 2^-100 to 2^100 against infinite weights, and one by one against finite ones: their three terms are
    exact, so a product of 8 bits more is off by its roundings only, one per term."""
    ctx, K = gpu
    g, L, m, k = np.random.default_rng(bits), ai.linear_weight, 201, 64
    top = g.integers(2 ** (bits - 1), 2 ** bits, (m, k)).astype(np.float64)
    top[:, :4] = 2.0 ** (bits - 1), 2.0 ** bits - 1, 2.0 ** (bits - 1), 2.0 ** bits - 1
    x = top * np.where(g.random((m, k)) < 0.5, -1.0, 1.0) * 2.0 ** (np.arange(-100, 101) - bits + 1.0)[:, None]
    assert np.array_equal(x, x.astype(np.float32))
    w = np.zeros((2 * k, k))
    w[np.arange(k), np.arange(k)], w[k + np.arange(k), np.arange(k)] = np.inf, M.rounded(g.standard_normal(k))
    out, batch = empty(ai, ctx, m * 2 * k, ai.F32), ai.CommandBatch(ctx)
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(2 * k)])
    print(f"small terms {bits}", flush=True)
    lin.rows_into(batch, K, upload(ai, ctx, x, ai.F32), ai.F32, m, [out], ai.F32)
    batch.commit_and_wait()
    got, want = download(ai, out, m * 2 * k, ai.F32).reshape(m, 2 * k), x * w[k:].sum(1)
    assert np.array_equal(got[:, :k], np.sign(x) * np.inf)
    assert (np.abs(got[:, k:] - want) <= 3 * 2.0 ** -24 * np.abs(want)).all()


@pytest.mark.parametrize("m,pos,k,heads,dim,pad,vdim", [(2048, 0, 64, 8, 128, 128, 128), (1500, 32, 128, 8, 96, 128, 160), (1500, 5, 64, 8, 96, 128, 160),
                                                        (1100, 64, 64, 12, 80, 96, 144), (130, 32, 64, 2, 32, 32, 64), (300, 0, 128, 3, 40, 64, 96), (64, 96, 72, 2, 32, 32, 64)])
def test_caches_of_many_rows(ai, gpu, m, pos, k, heads, dim, pad, vdim):
    """Whole and partial blocks of 32 positions of the value cache, padded keys at a position and a gated pair layout from products of many rows."""
    ctx, K = gpu
    g, L, cap = np.random.default_rng(pos + m), ai.linear_weight, (pos + m + 40) // 32 * 32
    ws = [M.rounded(g.standard_normal((heads * d, k)) / np.sqrt(k)) for d in (dim, dim, vdim)]
    x = M.rounded(g.standard_normal((m, k)))
    b = [g.standard_normal(w.shape[0]).astype(np.float32) for w in ws]
    lin = L.StackedLinear(ctx, [M.bf16_bits(w) for w in ws], [L.Segment(heads * dim, ai.ACT_SILU, dim, pad), L.Segment(heads * dim, 0, dim, pad, ai.ROWS_AT_POSITION),
                                                              L.Segment(heads * vdim, 0, vdim, vdim, ai.BLOCKS_AT_POSITION)], b)
    q, kc, v = (empty(ai, ctx, c, ai.BF16) for c in (m * heads * pad, cap * heads * pad, cap * heads * vdim))
    print(f"caches {m} {pos} {k}", flush=True)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, upload(ai, ctx, x, ai.BF16), ai.BF16, m, [q, kc, v], ai.BF16, ai.Buffer.from_slice(ctx, np.array([pos], np.uint32)))
    pairs = L.StackedLinear(ctx, [M.bf16_bits(ws[0])], [L.Segment(heads * dim, ai.ACT_SILU_PAIRS)])
    h = empty(ai, ctx, m * heads * dim // 2, ai.BF16)
    pairs.rows_into(batch, K, upload(ai, ctx, x, ai.BF16), ai.BF16, m, [h], ai.BF16)
    batch.commit_and_wait()
    got = download(ai, q, m * heads * pad, ai.BF16).reshape(m, heads, pad)
    close(got[:, :, :dim], O.silu(x @ ws[0].T + b[0]).reshape(m, heads, dim), BF16_TOL, "q")
    assert not got[:, :, dim:].any()
    got = download(ai, kc, cap * heads * pad, ai.BF16).reshape(cap, heads, pad)
    close(got[pos:pos + m, :, :dim], (x @ ws[1].T + b[1]).reshape(m, heads, dim), BF16_TOL, "k")
    assert not got[:pos].any() and not got[pos + m:].any() and not got[:, :, dim:].any()
    got = values_from_cache(download(ai, v, cap * heads * vdim, ai.BF16), heads * vdim)
    close(got[pos:pos + m], x @ ws[2].T + b[2], BF16_TOL, "v")
    assert not got[:pos].any() and not got[pos + m:].any()
    z = (x @ ws[0].T).reshape(m, -1, 2)
    close(download(ai, h, m * heads * dim // 2, ai.BF16).reshape(m, -1), O.silu(z[:, :, 0]) * z[:, :, 1], BF16_TOL, "pairs")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("m,pos,width,heads,dim,pad,vdim,vpad", [(5, 30, 64, 3, 20, 32, 12, 32), (1, 31, 64, 3, 20, 32, 12, 32), (70, 1, 40, 2, 32, 32, 64, 64),
                                                                 (1, 32, 520, 1, 5, 32, 33, 64), (33, 63, 36, 2, 24, 32, 40, 64), (40, 100, 64, 2, 16, 32, 32, 32)])
def test_segments_write_caches_at_the_position(ai, gpu, dtype, m, pos, width, heads, dim, pad, vdim, vpad):
    """Three segments: plain rows, padded heads at the position, value blocks at the position; rows past the end are dropped."""
    ctx, K = gpu
    dt = ai.BF16 if dtype == "bf16" else ai.F32
    g, L, cap = np.random.default_rng(pos + m), ai.linear_weight, 128
    ws = [M.rounded(g.standard_normal((heads * d, width)) / np.sqrt(width)) for d in (dim, dim, vdim)]
    x = stored(g.standard_normal((m, width)), ai, dt)
    b = [g.standard_normal(w.shape[0]).astype(np.float32) for w in ws]
    lin = L.StackedLinear(ctx, [M.bf16_bits(w) for w in ws],
                          [L.Segment(heads * dim, ai.ACT_SILU, dim, pad), L.Segment(heads * dim, 0, dim, pad, ai.ROWS_AT_POSITION),
                           L.Segment(heads * vdim, 0, vdim, vpad, ai.BLOCKS_AT_POSITION)], b)
    q, k, v = empty(ai, ctx, m * heads * pad, dt), empty(ai, ctx, cap * heads * pad, dt), empty(ai, ctx, cap * heads * vpad, dt)
    p = ai.Buffer.from_slice(ctx, np.array([pos], np.uint32))
    print(f"segments {dtype} {m} {pos}", flush=True)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, upload(ai, ctx, x, dt), dt, m, [q, k, v], dt, p)
    batch.commit_and_wait()

    def check():
        tol = BF16_TOL if dt == ai.BF16 else F32_TOL
        got = download(ai, q, m * heads * pad, dt).reshape(m, heads, pad)
        close(got[:, :, :dim], O.silu(x @ ws[0].T + b[0]).reshape(m, heads, dim), tol, "q")
        assert not got[:, :, dim:].any()
        stay = min(m, cap - pos)
        got = download(ai, k, cap * heads * pad, dt).reshape(cap, heads, pad)
        close(got[pos:pos + stay, :, :dim], (x @ ws[1].T + b[1]).reshape(m, heads, dim)[:stay], tol, "k")
        assert not got[:pos].any() and not got[pos + stay:].any() and not got[:, :, dim:].any()
        got = values_from_cache(download(ai, v, cap * heads * vpad, dt), heads * vpad).reshape(cap, heads, vpad)
        close(got[pos:pos + stay, :, :vdim], (x @ ws[2].T + b[2]).reshape(m, heads, vdim)[:stay], tol, "v")
        assert not got[:pos].any() and not got[pos + stay:].any() and not got[:, :, vdim:].any()
    check()
    if m == 1:
        for t in (q, k, v):
            t.fill_zero()
        K.linear_vector_into(batch, upload(ai, ctx, x, dt), dt, lin.weight, lin.bias, width, lin.segments, [q, k, v], dt, False, p)
        batch.commit_and_wait()
        check()


@pytest.mark.parametrize("sizes,blocks", [((16, 32, 16), 1), ((8, 8, 16), 1), ((32, 16, 16), 0), ((16, 16, 32), 2), ((96, 32, 64, 64), 1), ((48, 16, 32, 160), 2)])
@pytest.mark.parametrize("m,k", [(20, 64), (40, 64), (32800, 72), (65600, 72), (24640, 64), (32800, 64), (65600, 64)])
def test_value_blocks_among_other_segments(ai, gpu, sizes, blocks, m, k):
    """A value cache's segment before, between and behind others, narrower than the columns that a wave finishes at once, on every tile
    size (32 to 256 rows; 200 columns and more take the wide ones)."""
    ctx, K = gpu
    g, L, pos, cap, few = np.random.default_rng(m + k + sum(sizes)), ai.linear_weight, 32, m // 32 * 32 + 64, min(m, 1000)
    w, x = M.rounded(g.standard_normal((sum(sizes), k)) / np.sqrt(k)), M.rounded(g.standard_normal((few, k)))
    rows = np.arange(m) % few
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(sum(sizes))])
    segments = L.Segments([L.Segment(n, 0, 0, 0, ai.BLOCKS_AT_POSITION if i == blocks else ai.ROWS) for i, n in enumerate(sizes)])
    outs = [empty(ai, ctx, (cap if i == blocks else m) * n, ai.BF16) for i, n in enumerate(sizes)]
    print(f"blocks among segments {sizes} {blocks} {m} {k}", flush=True)
    batch = ai.CommandBatch(ctx)
    lin.rows_into(batch, K, ai.Buffer.from_slice(ctx, M.bf16_bits(x)[rows]), ai.BF16, m, outs, ai.BF16, ai.Buffer.from_slice(ctx, np.array([pos], np.uint32)), segments)
    batch.commit_and_wait()
    want, at = x @ w.T, 0
    for i, n in enumerate(sizes):
        got = download(ai, outs[i], (cap if i == blocks else m) * n, ai.BF16)
        if i == blocks:
            got = values_from_cache(got, n)
            assert not got[:pos].any() and not got[pos + m:].any()
            got = got[pos:pos + m]
        close(got.reshape(m, n), want[rows, at:at + n], BF16_TOL, f"segment {i}")
        at += n


@pytest.mark.parametrize("k,n", [(64, 40), (60, 33), (512, 130), (1000, 64), (1536, 20), (4096, 70), (9000, 12), (2501, 9)])
def test_linear_vector_stages(ai, gpu, k, n):
    """The norm (with an addition and a stored sum) and the gated norm in front of a one-row product."""
    ctx, K = gpu
    g, L, eps = np.random.default_rng(k), ai.linear_weight, 1e-3
    w = M.rounded(g.standard_normal((n, k)) / np.sqrt(k))
    x, add, nw, gate = (stored(g.standard_normal(k), ai, ai.F32) for _ in range(4))
    lin = L.StackedLinear(ctx, [M.bf16_bits(w)], [L.Segment(n)])
    xb, ab, nb = (upload(ai, ctx, t, ai.F32) for t in (x, add, nw))
    print(f"vector stages {k} {n}", flush=True)
    batch = ai.CommandBatch(ctx)
    outs = [empty(ai, ctx, n, ai.F32) for _ in range(4)]
    kept = empty(ai, ctx, k, ai.F32)
    lin.normed_vector_into(batch, K, xb, nb, eps, [outs[0]], ai.F32)
    lin.normed_vector_into(batch, K, xb, nb, eps, [outs[1]], ai.F32, None, ab, kept)
    for i, dt in ((2, ai.F32), (3, ai.BF16)):
        K.linear_gated_vector_into(batch, xb, upload(ai, ctx, gate, dt), dt, nb, eps, lin.weight, None, k, lin.segments, [outs[i]], ai.F32)
    batch.commit_and_wait()
    got = [download(ai, o, n, ai.F32) for o in outs]
    close(got[0], w @ (O.unit_rms(x, eps) * nw), F32_TOL)
    close(got[1], w @ (O.unit_rms(x + add, eps) * nw), F32_TOL)
    close(download(ai, kept, k, ai.F32), x + add, F32_TOL)
    close(got[2], w @ (O.unit_rms(x, eps) * nw * O.sigmoid(gate)), F32_TOL)
    close(got[3], w @ (O.unit_rms(x, eps) * nw * O.sigmoid(M.rounded(gate))), F32_TOL)
    with pytest.raises(ai.InvalidArgument):          # the sum must not go where the other workgroups still read
        lin.normed_vector_into(batch, K, xb, nb, eps, [outs[0]], ai.F32, None, ab, xb)


@pytest.mark.parametrize("k,n", [(8, 2047), (8, 2049), (520, 4098), (1024, 8200), (1032, 6145), (2048, 10250), (2056, 4097), (4096, 2060), (16, 140000),
                                 (4104, 258), (4160, 770), (8192, 1290), (8200, 515), (16384, 1030), (4104, 16390)])
@pytest.mark.parametrize("pairs", [False, True])
def test_one_row_walks(ai, gpu, k, n, pairs):
    """One row times more weight rows than there are waves: each takes none to six of them or more than a wave has lanes, with an
    addition to what the output held, and in pairs."""
    ctx, K = gpu
    g, L = np.random.default_rng(k + n), ai.linear_weight
    n += n % 2 if pairs else 0
    some = M.rounded(g.standard_normal((min(n, 1009), k)) / np.sqrt(k))
    x, pick, b = stored(g.standard_normal(k), ai, ai.F32), np.arange(n) % len(some), g.standard_normal(n).astype(np.float32)
    want = (some @ x)[pick] + b
    lin = L.StackedLinear(ctx, [M.bf16_bits(some)[pick]], [L.Segment(n, ai.ACT_SILU_PAIRS if pairs else ai.ACT_NONE)], [b])
    print(f"one row {k} {n} {pairs}", flush=True)
    if pairs:
        want = want[0::2] * O.sigmoid(want[0::2]) * want[1::2]
    out, res, batch = empty(ai, ctx, len(want), ai.F32), upload(ai, ctx, np.ones(n), ai.F32), ai.CommandBatch(ctx)
    xb = upload(ai, ctx, x, ai.F32)
    lin.vector_into(batch, K, xb, ai.F32, [out], ai.F32)
    if not pairs:
        K.linear_vector_into(batch, xb, ai.F32, lin.weight, lin.bias, k, lin.segments, [res], ai.F32, True)
    batch.commit_and_wait()
    close(download(ai, out, len(want), ai.F32), want, F32_TOL, "stored")
    if not pairs:
        close(download(ai, res, n, ai.F32), want + 1, F32_TOL, "added")


@pytest.mark.parametrize("k,n", [(8, 1), (512, 2048), (520, 2046), (2048, 2048), (2048, 33), (2056, 1), (2064, 2047), (3000, 300), (4088, 1030), (4096, 2048)])
@pytest.mark.parametrize("pairs", [False, True])
def test_one_row_against_few_rows(ai, gpu, k, n, pairs):
    """The same up to eight weight rows per CU: workgroups of four waves, and a row over eight waves beyond 2048 columns."""
    test_one_row_walks(ai, gpu, k, n, pairs)


@pytest.mark.parametrize("rows,dim", [(1, 64), (5, 100), (3, 1024), (2, 4096), (4, 5000), (70, 33)])
def test_row_norms_and_gather(ai, gpu, rows, dim):
    ctx, K = gpu
    g, eps = np.random.default_rng(dim), 1e-4
    x, add, gate = (stored(g.standard_normal((rows, dim)), ai, ai.F32) for _ in range(3))
    w = stored(g.standard_normal(dim), ai, ai.F32)
    xb, ab, wb = upload(ai, ctx, x, ai.F32), upload(ai, ctx, add, ai.F32), upload(ai, ctx, w, ai.F32)
    batch = ai.CommandBatch(ctx)
    print(f"norms {rows} {dim}", flush=True)
    for dt, tol in ((ai.F32, F32_TOL), (ai.BF16, BF16_TOL)):
        out, kept, picked = empty(ai, ctx, rows * dim, dt), empty(ai, ctx, rows * dim, ai.F32), empty(ai, ctx, 3 * dim, dt)
        K.norm_rows_f32_into(batch, xb, ab, wb, kept, None, out, dt, dim, rows, eps)
        pick = [rows - 1, 0, rows // 2]
        K.norm_rows_f32_into(batch, xb, None, wb, None, ai.Buffer.from_slice(ctx, np.array(pick, np.uint32)), picked, dt, dim, 3, eps)
        gated = empty(ai, ctx, rows * dim, dt)
        K.gated_norm_rows_into(batch, xb, upload(ai, ctx, gate, dt), wb, gated, dt, dim, rows, eps)
        batch.commit_and_wait()
        close(download(ai, out, rows * dim, dt).reshape(rows, dim), O.unit_rms(x + add, eps) * w, tol)
        close(download(ai, kept, rows * dim, ai.F32).reshape(rows, dim), x + add, F32_TOL)
        close(download(ai, picked, 3 * dim, dt).reshape(3, dim), (O.unit_rms(x, eps) * w)[pick], tol)
        close(download(ai, gated, rows * dim, dt).reshape(rows, dim), O.unit_rms(x, eps) * w * O.sigmoid(stored(gate, ai, dt)), tol)
    table = g.standard_normal((9, dim))
    idx = np.array([8, 0, 3, 200], np.uint32)
    out = empty(ai, ctx, 4 * dim, ai.F32)
    K.embed_rows_bf16_into(batch, upload(ai, ctx, table, ai.BF16), 9, dim, ai.Buffer.from_slice(ctx, idx), 4, out)
    z = x.astype(np.float32)
    z[0, dim // 2] = z[0, dim - 1] = 9.0
    best, pos = ai.Buffer.empty(ctx, 4 * rows), ai.Buffer.from_slice(ctx, np.array([5], np.uint32))
    K.argmax_rows_f32_into(batch, ai.Buffer.from_slice(ctx, z), best, rows, dim)
    K.advance_position_into(batch, pos, 7)
    batch.commit_and_wait()
    assert np.array_equal(download(ai, out, 4 * dim, ai.F32).reshape(4, dim), M.rounded(table)[[8, 0, 3, 8]])
    assert best.as_array(np.uint32).tolist() == z.argmax(1).tolist() and pos.as_array(np.uint32, 1)[0] == 12


# ---- softmax attention -------------------------------------------------------------------------------------------------
def attention_case(ai, gpu, dtype, maps, heads, kv_heads, dim, vdim, start, rows, cap, seed=0, spike=None, stale=False, lam=0.4, out_scale=0.7, poison=(), scale=None):
    """Caches filled as the projections fill them.  `spike` = (row, key): one key that takes nearly all of a row's weight."""
    ctx, K = gpu
    dt = ai.BF16 if dtype == "bf16" else ai.F32
    g, eps, scale = np.random.default_rng(seed + start + rows + dim), 1e-5, dim ** -0.5 if scale is None else scale
    L, dq, dv = start + rows, K.attention_padded_dim(dim), K.attention_padded_vdim(vdim)
    q, k, v = (stored(g.standard_normal(s), ai, dt) for s in ((rows, heads, maps, dim), (L, kv_heads, maps, dim), (L, kv_heads, vdim)))
    if spike is not None:
        row, key = spike
        u = np.sign(g.standard_normal(dim))
        k[key] = stored(u * 5.0, ai, dt)
        q[row] = stored(u * 14.0 / np.sqrt(dim), ai, dt)
    fill = 3.0 if stale else 0.0                      # what an earlier, longer sequence would have left behind
    kc, vc, qp = np.full((cap, kv_heads, maps, dq), fill), np.full((cap, kv_heads, dv), fill), np.zeros((rows, heads, maps, dq))
    kc[:, :, :, dim:] = vc[:, :, vdim:] = 0.0
    kc[:L, :, :, :dim], vc[:L, :, :vdim], qp[..., :dim] = k, v, q
    for key, column, value in poison:
        vc[key, :, column] = value
    blocks = np.zeros((cap // 32, kv_heads * dv, 32))
    blocks[:, :, block_order()] = vc.reshape(cap // 32, 32, kv_heads * dv).transpose(0, 2, 1)
    out, pos = empty(ai, ctx, rows * heads * vdim, dt), ai.Buffer.from_slice(ctx, np.array([start], np.uint32))
    print(f"attention {dtype} maps {maps} heads {heads}/{kv_heads} dim {dim} vdim {vdim} start {start} rows {rows}", flush=True)
    batch = ai.CommandBatch(ctx)
    K.attention_rows_into(batch, upload(ai, ctx, qp, dt), upload(ai, ctx, kc, dt), upload(ai, ctx, blocks, dt), out, dt, pos, start, rows, heads,
                          kv_heads, maps, dim, vdim, cap, scale, lam, out_scale, eps)
    batch.commit_and_wait()
    got = download(ai, out, rows * heads * vdim, dt).reshape(rows, heads, vdim)
    if poison:
        return got
    want = np.zeros((rows, heads, vdim))
    for h in range(heads):
        j = h // (heads // kv_heads)
        a = [O.causal_softmax_attention(q[:, h, m], k[:, j, m], v[:, j], scale, start) for m in range(maps)]
        want[:, h] = a[0] if maps == 1 else O.unit_rms(a[0] - lam * a[1], eps) * out_scale
    # over a thousand random keys the difference of the two averages is small and its norm enlarges the rounding of both sums about thirtyfold
    close(got, want, BF16_TOL if dt == ai.BF16 else F32_TOL if maps == 1 else 1e-4, "attention")
    if spike is not None and maps == 1:
        close(got[spike[0]].reshape(kv_heads, -1, vdim), v[spike[1]][:, None].repeat(heads // kv_heads, 1), 0.03, "the far key's value")
    return got


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(3, 3, 32, 64), (6, 2, 24, 40), (8, 1, 64, 128), (3, 3, 8, 16), (4, 2, 128, 256), (5, 1, 20, 33), (34, 2, 16, 24)])
@pytest.mark.parametrize("start,rows", [(0, 1), (31, 1), (32, 2), (95, 34), (0, 97), (63, 190), (0, 64), (1, 64)])
def test_attention_shapes(ai, gpu, dtype, maps, heads, kv_heads, dim, vdim, start, rows):
    attention_case(ai, gpu, dtype, maps, heads, kv_heads, dim, vdim, start, rows, 256)


@pytest.mark.parametrize("dim,vdim", [(32, 32), (32, 128), (32, 256), (64, 32), (64, 64), (64, 256), (128, 32), (128, 64), (128, 128), (128, 256), (136, 64), (48, 300)])
@pytest.mark.parametrize("rows", [1, 150])
@pytest.mark.parametrize("maps", [1, 2])
def test_attention_every_head_size(ai, gpu, maps, dim, vdim, rows):
    attention_case(ai, gpu, "bf16", maps, 4, 2, dim, vdim, 70, rows, 256)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rows", [1, 3, 300])
@pytest.mark.parametrize("key", [0, 1, 31, 32, 33, 511, 1000, 1023])
def test_attention_finds_one_key_far_away(ai, gpu, dtype, rows, key):
    attention_case(ai, gpu, dtype, 1, 4, 2, 32, 64, 1023, rows, 1344, spike=(rows - 1, key))
    attention_case(ai, gpu, dtype, 2, 4, 2, 32, 64, 1023, rows, 1344, spike=(0, key))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("heads,kv_heads,maps,dim,vdim", [(16, 1, 2, 64, 128), (17, 1, 1, 64, 128), (4, 4, 1, 192, 256), (6, 3, 2, 40, 30)])
@pytest.mark.parametrize("start", [0, 255, 256, 638, 639, 640])
def test_attention_of_one_row(ai, gpu, dtype, heads, kv_heads, maps, dim, vdim, start):
    """One block of keys, one and two a wave, the longest context that a workgroup takes of narrow positions and the next (of wide ones: the test below);
    sixteen heads a kv head and seventeen."""
    attention_case(ai, gpu, dtype, maps, heads, kv_heads, dim, vdim, start, 1, (start + 32) // 32 * 32)


@pytest.mark.parametrize("heads,kv_heads,maps,dim,vdim,alone,split", [(8, 2, 1, 64, 64, [638], [639]), (16, 4, 2, 64, 128, [606], [607]), (8, 2, 1, 128, 128, [606], [607]),
                                                                      (8, 2, 1, 192, 128, [350, 383, 478], [351, 382, 479]), (4, 2, 2, 128, 128, [350], [351, 382, 511]),
                                                                      (8, 1, 1, 192, 256, [255, 350], [351, 638])])
def test_attention_of_one_row_by_the_columns_of_a_position(ai, gpu, heads, kv_heads, maps, dim, vdim, alone, split):
    """Wide rows are read by many workgroups from fewer keys on: one launch up to a line, two behind it."""
    ctx, K = gpu
    b = ai.Buffer.empty(ctx, 672 * kv_heads * (maps * 192 + 256) * 2)
    b.fill_zero()
    for start in alone + split:
        attention_case(ai, gpu, "bf16", maps, heads, kv_heads, dim, vdim, start, 1, (start + 32) // 32 * 32)
        batch = ai.CommandBatch(ctx)
        K.attention_rows_into(batch, b, b, b, ai.Buffer.empty(ctx, heads * vdim * 2), ai.BF16, b, start, 1, heads, kv_heads, maps, dim, vdim, 672, 1.0, 0.4, 0.7, 1e-5)
        assert batch.dispatch_count() == (1 if start in alone else 2), start
        batch.commit_and_wait()


@pytest.mark.parametrize("rows", [1, 40, 200])
def test_attention_ignores_what_lies_behind_the_last_position(ai, gpu, rows):
    """Stale rows and block entries past the last position (a slot that is used again) must not change a bit."""
    a = attention_case(ai, gpu, "bf16", 2, 4, 2, 32, 64, 45, rows, 320)
    b = attention_case(ai, gpu, "bf16", 2, 4, 2, 32, 64, 45, rows, 320, stale=True)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("dim,vdim", [(32, 32), (20, 33), (64, 64), (33, 128), (128, 128), (100, 256), (136, 64), (192, 128), (200, 250), (256, 256)])
@pytest.mark.parametrize("start,rows", [(0, 1), (70, 1), (31, 18), (5, 150)])
@pytest.mark.parametrize("maps", [1, 2])
def test_wide_attention_every_head_size(ai, gpu, maps, dim, vdim, start, rows):
    a = attention_case(ai, gpu, "f32", maps, 4, 2, dim, vdim, start, rows, 256)
    assert np.array_equal(a, attention_case(ai, gpu, "f32", maps, 4, 2, dim, vdim, start, rows, 256, stale=True))


@pytest.mark.parametrize("dim,vdim", [(32, 32), (64, 64), (33, 128), (128, 256)])
@pytest.mark.parametrize("start,rows", [(0, 40), (31, 18), (70, 50)])
@pytest.mark.parametrize("maps", [1, 2])
def test_wide_attention_rows_do_not_see_what_follows(ai, gpu, maps, dim, vdim, start, rows):
    """An infinity or NaN among the values reaches its column of the rows from its position on, and nothing else: that stays as it is up to
    the order of the f32 sums (F32_TOL with one map; the norm behind two enlarges it)."""
    keys = (start + 5, start + 14, start + rows - 1)
    clean = attention_case(ai, gpu, "f32", maps, 4, 2, dim, vdim, start, rows, 256)
    got = attention_case(ai, gpu, "f32", maps, 4, 2, dim, vdim, start, rows, 256, poison=[(keys[0], 3, np.inf), (keys[1], vdim - 1, np.nan), (keys[2], 7, -np.inf)])
    close(got[:5], clean[:5], F32_TOL if maps == 1 else 1e-4, "rows before")
    if maps == 1:
        for t in range(rows):
            special = {3: np.inf} if t >= 5 else {}
            if t >= rows - 1:
                special[7] = -np.inf
            for c in range(vdim):
                if c == vdim - 1 and t >= 14:
                    assert np.isnan(got[t, :, c]).all()
                elif c in special:
                    assert (got[t, :, c] == special[c]).all()
                else:
                    assert np.abs(got[t, :, c] - clean[t, :, c]).max() <= F32_TOL * np.abs(clean).max(), (t, c)


def test_attention_long_context_splits(ai, gpu):
    for rows in (1, 5):
        attention_case(ai, gpu, "bf16", 2, 2, 1, 32, 32, 9000, rows, 9056, spike=(0, 37))


@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("dim,vdim,heads,start,rows", [(32, 32, 4, 1023, 300), (64, 33, 4, 1500, 260), (20, 128, 8, 700, 129), (128, 250, 4, 1023, 257),
                                                       (32, 64, 16, 0, 1300), (64, 128, 16, 40, 700)])
def test_attention_of_many_rows(ai, gpu, maps, dim, vdim, heads, start, rows):
    """A few splits of many rows, and launches whose workgroups are all on the chip at once, two a CU."""
    attention_case(ai, gpu, "bf16", maps, heads, 2 if heads < 16 else 4, dim, vdim, start, rows, (start + rows + 31) // 32 * 32)


@pytest.mark.parametrize("scale", [-0.2, 0.0])
@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("dtype,heads,kv_heads,dim,vdim,start,rows", [("bf16", 4, 2, 32, 64, 50, 20), ("bf16", 8, 2, 64, 128, 40, 150), ("bf16", 4, 4, 24, 40, 100, 90),
                                                                     ("f32", 4, 2, 32, 64, 50, 20), ("f32", 4, 2, 64, 64, 40, 1)])
def test_attention_scales_of_zero_and_below(ai, gpu, scale, maps, dtype, heads, kv_heads, dim, vdim, start, rows):
    """Whose sign, or that they are zero, goes into the queries: up to 64 rows of a key head and tiles of more."""
    attention_case(ai, gpu, dtype, maps, heads, kv_heads, dim, vdim, start, rows, (start + rows + 31) // 32 * 32, scale=scale)


def test_attention_rejects(ai, gpu):
    ctx, K = gpu
    b, batch = ai.Buffer.empty(ctx, 1 << 16), ai.CommandBatch(ctx)
    for args in ((5, 1, 3, 2, 1, 32, 32, 32), (31, 2, 2, 2, 1, 32, 32, 32), (0, 1, 2, 2, 3, 32, 32, 32), (0, 1, 2, 2, 1, 32, 32, 40)):
        with pytest.raises(ai.InvalidArgument):
            K.attention_rows_into(batch, b, b, b, b, ai.BF16, b, *args, 1.0)
    assert batch.dispatch_count() == 0


# ---- linear attention --------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("dim", [5, 32, 40, 64, 100, 128, 200, 300, 512, 700, 1024])
@pytest.mark.parametrize("rows", [7, 8, 9, 17, 40])
def test_recurrence_over_rows(ai, gpu, dtype, dim, rows):
    """Around the number of rows whose inputs are on their way together, for every number of state values a lane holds."""
    ctx, K = gpu
    dt = ai.BF16 if dtype == "bf16" else ai.F32
    g, H, vdim = np.random.default_rng(dim + rows), 2, 19
    dq = K.linear_attention_padded_dim(dim)
    q, k, v = (stored(g.standard_normal(s) / np.sqrt(dim), ai, dt) for s in ((rows, H, dim), (rows, H, dim), (rows, H, vdim)))
    decay, S = np.array([0.5, 0.97], np.float32), g.standard_normal((H, dim, vdim)).astype(np.float32)
    pad = np.full((rows, H, dq), 7.0)                  # what pads a row is not read
    qp, kp = pad.copy(), pad.copy()
    qp[..., :dim], kp[..., :dim] = q, k
    state = np.zeros((H, vdim, dq), np.float32)
    state[:, :, :dim] = S.transpose(0, 2, 1)
    st, out = ai.Buffer.from_slice(ctx, state), empty(ai, ctx, rows * H * vdim, ai.F32)
    print(f"recurrence {dtype} {dim} {rows}", flush=True)
    batch = ai.CommandBatch(ctx)
    K.linear_attention_recurrent_into(batch, upload(ai, ctx, qp, dt), upload(ai, ctx, kp, dt), upload(ai, ctx, v, dt), dt, st, ai.Buffer.from_slice(ctx, decay), out,
                                      rows, H, dim, vdim, 0.5)
    batch.commit_and_wait()
    want, end = O.lightning_recurrence(q, k, v, decay.astype(np.float64), S.astype(np.float64))
    close(download(ai, out, rows * H * vdim, ai.F32).reshape(rows, H, vdim), 0.5 * want, F32_TOL, "output")
    got = st.as_array(np.float32, H * vdim * dq).reshape(H, vdim, dq)
    close(got[:, :, :dim], end.transpose(0, 2, 1), F32_TOL, "state")
    assert not got[:, :, dim:].any()


@pytest.mark.parametrize("heads,vdim,dim", [(16, 128, 128), (41, 50, 128), (41, 50, 100), (33, 64, 65), (17, 128, 160)])
@pytest.mark.parametrize("rows", [1, 7, 8, 33])
def test_recurrence_of_many_columns(ai, gpu, heads, vdim, dim, rows):
    """Around the columns beyond which many rows share a wave's lanes, with fixed decays and with a head's steps computed from the token."""
    ctx, K = gpu
    g = np.random.default_rng(heads + dim + rows)
    dq = K.linear_attention_padded_dim(dim)
    q, k, v = (M.rounded(g.standard_normal(s) / np.sqrt(dim)) for s in ((rows, heads, dim), (rows, heads, dim), (rows, heads, vdim)))
    decay, S = np.linspace(0.4, 1.0, heads).astype(np.float32), g.standard_normal((heads, dim, vdim)).astype(np.float32)
    qp, kp = np.full((rows, heads, dq), 3.0), np.full((rows, heads, dq), 3.0)
    qp[..., :dim], kp[..., :dim] = q, k
    state = np.zeros((heads, vdim, dq), np.float32)
    state[:, :, :dim] = S.transpose(0, 2, 1)
    for dt in (ai.BF16, ai.F32):
        st, out = ai.Buffer.from_slice(ctx, state), empty(ai, ctx, rows * heads * vdim, ai.F32)
        batch = ai.CommandBatch(ctx)
        K.linear_attention_recurrent_into(batch, upload(ai, ctx, qp, dt), upload(ai, ctx, kp, dt), upload(ai, ctx, v, dt), dt, st, ai.Buffer.from_slice(ctx, decay), out,
                                          rows, heads, dim, vdim, 0.5)
        batch.commit_and_wait()
        want, end = O.lightning_recurrence(q, k, v, decay.astype(np.float64), S.astype(np.float64))
        close(download(ai, out, rows * heads * vdim, ai.F32).reshape(rows, heads, vdim), 0.5 * want, F32_TOL, "output")
        got = st.as_array(np.float32, heads * vdim * dq).reshape(heads, vdim, dq)
        close(got[:, :, :dim], end.transpose(0, 2, 1), F32_TOL, "state")
        assert not got[:, :, dim:].any()


@pytest.mark.parametrize("heads,vdim,dim", [(16, 128, 128), (41, 50, 128), (41, 50, 100), (33, 64, 65), (17, 128, 160), (40, 128, 160), (81, 64, 256), (44, 117, 129), (3, 50, 300)])
@pytest.mark.parametrize("rows", [1, 7, 8, 11, 12, 23, 24, 33])
def test_recurrence_of_few_and_of_many_columns(ai, gpu, heads, vdim, dim, rows):
    """Around the columns beyond which many rows share a wave's lanes, and the rows at which it has more of them ahead, with fixed decays and with a
    head's steps computed from the token."""
    ctx, K = gpu
    g = np.random.default_rng(heads + dim + rows)
    dq = K.linear_attention_padded_dim(dim)
    q, k, v = (M.rounded(g.standard_normal(s) / np.sqrt(dim)) for s in ((rows, heads, dim), (rows, heads, dim), (rows, heads, vdim)))
    decay, S = np.linspace(0.4, 1.0, heads).astype(np.float32), g.standard_normal((heads, dim, vdim)).astype(np.float32)
    raw, (dt_bias, a_log, skip) = g.standard_normal((rows, heads)).astype(np.float32), g.standard_normal((3, heads)).astype(np.float32)
    qp, kp = np.full((rows, heads, dq), 3.0), np.full((rows, heads, dq), 3.0)
    qp[..., :dim], kp[..., :dim] = q, k
    state = np.zeros((heads, vdim, dq), np.float32)
    state[:, :, :dim] = S.transpose(0, 2, 1)
    for dt in (ai.BF16, ai.F32):
        buffers = [upload(ai, ctx, x, dt) for x in (qp, kp, v)]
        for selective in (False, True):
            st, out = ai.Buffer.from_slice(ctx, state), empty(ai, ctx, rows * heads * vdim, ai.F32)
            batch = ai.CommandBatch(ctx)
            if selective:
                K.selective_recurrent_into(batch, buffers[2], buffers[1], buffers[0], dt, *(ai.Buffer.from_slice(ctx, x) for x in (raw, dt_bias, a_log, skip)), st, out,
                                           rows, heads, vdim, heads, dim)
                want, end = O.selective_recurrence(v, k, q, O.softplus(raw.astype(np.float64) + dt_bias), a_log.astype(np.float64), skip.astype(np.float64), S.astype(np.float64))
            else:
                K.linear_attention_recurrent_into(batch, *buffers, dt, st, ai.Buffer.from_slice(ctx, decay), out, rows, heads, dim, vdim, 0.5)
                want, end = O.lightning_recurrence(q, k, v, decay.astype(np.float64), S.astype(np.float64))
                want = 0.5 * want
            batch.commit_and_wait()
            close(download(ai, out, rows * heads * vdim, ai.F32).reshape(rows, heads, vdim), want, F32_TOL, "output")
            got = st.as_array(np.float32, heads * vdim * dq).reshape(heads, vdim, dq)
            close(got[:, :, :dim], end.transpose(0, 2, 1), F32_TOL, "state")
            assert not got[:, :, dim:].any()


@pytest.mark.parametrize("heads,dim,vdim", [(4, 32, 48), (3, 20, 33), (2, 64, 128), (1, 128, 80), (2, 200, 48), (2, 8, 100)])
@pytest.mark.parametrize("cuts", [[1, 1, 1], [16, 2], [64], [17, 65, 130], [63, 1, 64], [300]])
def test_linear_attention_forms(ai, gpu, heads, dim, vdim, cuts):
    """Recurrent in both types and chunked, in portions: the outputs, and the state after every portion."""
    ctx, K = gpu
    g, T = np.random.default_rng(dim + sum(cuts)), sum(cuts)
    decay = np.array([0.9995, 0.3, 1.0, 0.0][:heads])
    dq = K.linear_attention_padded_dim(dim)
    q, k, v = (M.rounded(g.standard_normal(s)) for s in ((T, heads, dim), (T, heads, dim), (T, heads, vdim)))
    q[-1] = M.rounded(k[0] * 3)                      # the last row asks for the first
    for dt, chunked in ((ai.F32, False), (ai.BF16, False), (ai.BF16, True)):
        print(f"linear attention {heads} {dim} {vdim} {cuts} dtype {dt} chunked {chunked}", flush=True)
        state = ai.Buffer.empty(ctx, heads * vdim * dq * 4)
        db = ai.Buffer.from_slice(ctx, decay.astype(np.float32))
        pw = ai.Buffer.from_slice(ctx, (decay[:, None] ** np.arange(65)).astype(np.float32))
        s, at = None, 0
        for n in cuts:
            part = slice(at, at + n)
            qp, kp = np.full((n, heads, dq), 2.0), np.full((n, heads, dq), 2.0)      # the padding's content must not matter
            qp[..., :dim], kp[..., :dim] = q[part], k[part]
            qb, kb, vb = upload(ai, ctx, qp, dt), upload(ai, ctx, kp, dt), upload(ai, ctx, v[part], dt)
            out = empty(ai, ctx, n * heads * vdim, ai.F32)
            batch = ai.CommandBatch(ctx)
            if chunked:
                work = ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(n, heads, dim, vdim))
                K.linear_attention_chunked_into(batch, qb, kb, vb, state, pw, work, out, n, heads, dim, vdim)
            else:
                K.linear_attention_recurrent_into(batch, qb, kb, vb, dt, state, db, out, n, heads, dim, vdim)
            batch.commit_and_wait()
            want, s = O.lightning_recurrence(q[part], k[part], v[part], decay, s)
            close(download(ai, out, n * heads * vdim, ai.F32).reshape(n, heads, vdim), want, F32_TOL, f"rows {part}")
            got = state.as_array(np.float32).reshape(heads, vdim, dq)
            close(got[:, :, :dim].transpose(0, 2, 1), s, F32_TOL, f"state after {at + n}")
            at += n


@pytest.mark.parametrize("heads,dim,vdim,rows", [(64, 64, 64, 1100), (8, 256, 100, 1153), (3, 128, 64, 127), (3, 128, 64, 128), (2, 40, 6, 129), (2, 128, 130, 193),
                                                  (130, 20, 33, 127), (129, 32, 64, 128), (130, 64, 70, 193), (260, 8, 6, 129), (260, 40, 3, 130), (3, 20, 3, 70), (2, 200, 5, 64)])
def test_linear_attention_chunks(ai, gpu, heads, dim, vdim, rows):
    """Chunks of 128 rows (more than 256 workgroups with 64) and of 64: whole, one row short and over, ending in either half; one and several
    tiles of key and value columns, widths of values of all remainders."""
    ctx, K = gpu
    g = np.random.default_rng(heads + dim + rows)
    decay, dq = np.linspace(0.6, 1.0, heads), K.linear_attention_padded_dim(dim)
    q, k, v = (M.rounded(g.standard_normal(s)) for s in ((rows, heads, dim), (rows, heads, dim), (rows, heads, vdim)))
    pad = [(0, 0), (0, 0), (0, dq - dim)]
    state, out = ai.Buffer.empty(ctx, heads * vdim * dq * 4), empty(ai, ctx, rows * heads * vdim, ai.F32)
    pw = ai.Buffer.from_slice(ctx, (decay[:, None] ** np.arange(65)).astype(np.float32))
    work = ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(rows, heads, dim, vdim))
    print(f"chunks {heads} {dim} {vdim} {rows}", flush=True)
    batch = ai.CommandBatch(ctx)
    K.linear_attention_chunked_into(batch, upload(ai, ctx, np.pad(q, pad), ai.BF16), upload(ai, ctx, np.pad(k, pad), ai.BF16), upload(ai, ctx, v, ai.BF16), state, pw,
                                    work, out, rows, heads, dim, vdim)
    batch.commit_and_wait()
    want, end = O.lightning_recurrence(q, k, v, decay, None)
    close(download(ai, out, rows * heads * vdim, ai.F32).reshape(rows, heads, vdim), want, F32_TOL, "output")
    close(state.as_array(np.float32).reshape(heads, vdim, dq)[:, :, :dim], end.transpose(0, 2, 1), F32_TOL, "state")


@pytest.mark.parametrize("decay,rows", [(2.0, 17), (2.0, 100), (2.0, 127), (2.0, 130), (1.25, 200), (3.0, 70)])
@pytest.mark.parametrize("heads", [2, 130])
def test_linear_attention_decays_above_one(ai, gpu, decay, rows, heads):
    """Chunked: what is finite in steps of 64 rows is so; a row is judged against its own size, which grows with the decay's powers."""
    ctx, K = gpu
    g, dim, vdim = np.random.default_rng(rows), 32, 48
    q, k, v = (M.rounded(g.standard_normal(s)) for s in ((rows, heads, dim), (rows, heads, dim), (rows, heads, vdim)))
    k *= 2.0 ** -14
    decays = np.array([decay, 0.5] * (heads // 2))
    state, out = ai.Buffer.empty(ctx, heads * vdim * dim * 4), empty(ai, ctx, rows * heads * vdim, ai.F32)
    pw = ai.Buffer.from_slice(ctx, (decays[:, None] ** np.arange(65)).astype(np.float32))
    work = ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(rows, heads, dim, vdim))
    print(f"decays above one {decay} {rows}", flush=True)
    batch = ai.CommandBatch(ctx)
    K.linear_attention_chunked_into(batch, *(upload(ai, ctx, x, ai.BF16) for x in (q, k, v)), state, pw, work, out, rows, heads, dim, vdim)
    batch.commit_and_wait()
    want, end = O.lightning_recurrence(q, k, v, decays, None)
    size = np.abs(want).max(2, keepdims=True)
    close(download(ai, out, rows * heads * vdim, ai.F32).reshape(rows, heads, vdim).astype(np.float64) / size, want / size, F32_TOL, "output")
    got, size = state.as_array(np.float32).reshape(heads, vdim, dim).astype(np.float64), np.abs(end).max((1, 2))[:, None, None]
    close(got / size, end.transpose(0, 2, 1) / size, F32_TOL, "state")


def test_linear_attention_sums_are_rounded_little(ai, gpu):
    """Chunks of 128 rows against f64: no further off, in the 2-norm, than chunks of 64 rows with one running sum for all terms were (1.41e-7
    at this size, and 1.62e-7 with 128 rows)."""
    ctx, K = gpu
    g, rows, heads, dim, vdim = np.random.default_rng(3), 1024, 40, 32, 64
    q, k, v = (M.rounded(g.standard_normal((rows, heads, n))) for n in (dim, dim, vdim))
    decay = np.linspace(0.6, 0.9995, heads).astype(np.float32).astype(np.float64)
    state, out = ai.Buffer.empty(ctx, heads * vdim * dim * 4), empty(ai, ctx, rows * heads * vdim, ai.F32)
    pw, work = ai.Buffer.from_slice(ctx, (decay[:, None] ** np.arange(65)).astype(np.float32)), ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(rows, heads, dim, vdim))
    print("rounding of sums", flush=True)
    batch = ai.CommandBatch(ctx)
    K.linear_attention_chunked_into(batch, *(upload(ai, ctx, x, ai.BF16) for x in (q, k, v)), state, pw, work, out, rows, heads, dim, vdim)
    batch.commit_and_wait()
    t = np.arange(rows)
    between = np.maximum(t[:, None] - t, 0)
    want = np.stack([(q[:, h] @ k[:, h].T * np.tril(decay[h] ** between)) @ v[:, h] for h in range(heads)], 1)
    err = np.linalg.norm(download(ai, out, rows * heads * vdim, ai.F32).reshape(want.shape) - want) / np.linalg.norm(want)
    assert err <= 1.45e-7, err


def test_linear_attention_of_very_wide_rows(ai, gpu):
    """Rows of 2^24 values, which a chunk's 32-bit offsets do not reach, and a state of more than 2^32 bytes a head, which they do."""
    ctx, K = gpu
    g, rows = np.random.default_rng(1), 2
    heads, dim, vdim = 1 << 19, 32, 2
    q, k, v = (g.standard_normal((rows, heads, n)).astype(np.float32) for n in (dim, dim, vdim))
    q, k, v = ((x.view(np.uint32) & 0xFFFF0000).view(np.float32) for x in (q, k, v))      # bf16 values
    bits = lambda x: ai.Buffer.from_slice(ctx, (x.view(np.uint32) >> 16).astype(np.uint16))
    decay = g.uniform(0.5, 1.0, heads).astype(np.float32)
    state, out = ai.Buffer.empty(ctx, heads * vdim * dim * 4), empty(ai, ctx, rows * heads * vdim, ai.F32)
    pw, work = ai.Buffer.from_slice(ctx, decay[:, None] ** np.arange(65, dtype=np.float32)), ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(rows, heads, dim, vdim))
    print("very wide rows", flush=True)
    batch = ai.CommandBatch(ctx)
    K.linear_attention_chunked_into(batch, bits(q), bits(k), bits(v), state, pw, work, out, rows, heads, dim, vdim)
    batch.commit_and_wait()
    dot = lambda t, s: (q[t].astype(np.float64) * k[s]).sum(1)[:, None] * v[s]
    want = np.stack([dot(0, 0), decay[:, None] * dot(1, 0) + dot(1, 1)])
    close(download(ai, out, rows * heads * vdim, ai.F32).reshape(rows, heads, vdim), want, F32_TOL, "many heads")

    heads, dim, vdim, rows = 1, 256, (1 << 22) + 70, 3          # columns behind the offset at which 32 bits would begin again
    q, k = (M.rounded(g.standard_normal((rows, dim))) for _ in range(2))
    v, end = np.zeros((rows, vdim), np.float32), slice(vdim - 70, None)
    v[:, :70], v[:, end] = M.rounded(g.standard_normal((rows, 70))), M.rounded(g.standard_normal((rows, 70)))
    state, out = ai.Buffer.empty(ctx, vdim * dim * 4), empty(ai, ctx, rows * vdim, ai.F32)
    first = g.standard_normal((70, dim)).astype(np.float32)
    state.fill_zero()
    state.copy_from_bytes(first, offset=(vdim - 70) * dim * 4)
    pw, work = ai.Buffer.from_slice(ctx, (0.75 ** np.arange(65)).astype(np.float32)), ai.Buffer.empty(ctx, K.linear_attention_workspace_bytes(rows, heads, dim, vdim))
    print("a state of four gigabytes", flush=True)
    K.linear_attention_chunked_into(batch, upload(ai, ctx, q, ai.BF16), upload(ai, ctx, k, ai.BF16), upload(ai, ctx, v, ai.BF16), state, pw, work, out, rows, heads, dim, vdim)
    batch.commit_and_wait()
    got = download(ai, out, rows * vdim, ai.F32).reshape(rows, vdim)
    for part, begin in ((slice(0, 70), np.zeros((1, dim, 70))), (end, first.T[None].astype(np.float64))):
        want, _ = O.lightning_recurrence(q[:, None], k[:, None], v[:, None, part].astype(np.float64), np.array([0.75]), begin)
        close(got[:, part], want[:, 0], F32_TOL, f"columns {part}")


# ---- mixture of experts ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rows,experts,top,width,ff", [(9, 3, 2, 33, 20), (300, 2, 2, 1030, 24)])
def test_mixture_of_odd_widths(ai, gpu, dtype, rows, experts, top, width, ff):
    """Rows that are not made of 16-byte pieces."""
    test_mixture_of_experts(ai, gpu, dtype, rows, experts, top, width, ff)


@pytest.mark.parametrize("rows,experts,top,width,ff", [(1000, 5, 1, 2048, 1024), (770, 6, 2, 1024, 2048), (1600, 3, 1, 192, 4096), (400, 2, 1, 2048, 2048),
                                                       (2000, 4, 2, 2048, 1024), (4000, 2, 1, 2048, 1024), (4000, 8, 1, 2048, 512), (3500, 3, 1, 2048, 1024), (2000, 12, 1, 72, 1040)])
def test_mixture_of_large_experts(ai, gpu, rows, experts, top, width, ff):
    """Expert plans through the kernels of large products, by the rule for 256 CUs (first product / second): 1000 rows 64 x 64 / 128 x 128
    phased; 770, 1600 rows 256 x 128 phased / 64 x 64 and 32 x 32; 400 rows 64 x 64 with four buffers; 2000 rows with two
    of four experts and 4000 with one of two 256 x 128 / 256 x 256 phased, the second added up from slots and straight into the rows; 4000 with one of eight 128 x 128 / 256 x 256, 3500 128 x 128 / 256 x 128; 2000 of 12 128 x 128 of four waves / 32 x 32.
    Ragged last tiles, an expert with a few rows and one with none.  The reference is f32 arithmetic on the CPU."""
    ctx, K = gpu
    g = np.random.default_rng(rows + experts)
    x = M.rounded(g.standard_normal((rows, width))).astype(np.float32)
    ups, downs = (M.rounded(g.standard_normal(s) / np.sqrt(s[2])).astype(np.float32) for s in ((experts, ff, width), (experts, width, ff)))
    logits = g.standard_normal((rows, experts)).astype(np.float32)
    logits[:, 0] = -50.0                              # nobody's first choice but a few rows'
    logits[:7, 0] = 9.0
    if top == 1 and experts > 2:
        logits[:, 1] = -60.0
    order = np.argsort(-logits, axis=1, kind="stable")[:, :top]
    hidden_want, want = np.zeros((rows, top, ff), np.float32), np.zeros((rows, width), np.float32)
    for e in range(experts):
        t, c = np.nonzero(order == e)
        h = M.rounded(O.relu_squared(O.sigmoid(logits[t, e].astype(np.float64))[:, None] * (x[t] @ ups[e].T))).astype(np.float32)
        hidden_want[t, c] = h
        np.add.at(want, t, h @ downs[e].T)
    print(f"large experts {rows} {experts} {top} {width} {ff}", flush=True)
    plan = ai.Buffer.empty(ctx, 4 * K.moe_plan_words(rows, experts, top))
    up, down = (ai.Buffer.from_slice(ctx, M.bf16_bits(w)) for w in (ups, downs))
    hidden, slots, rb = empty(ai, ctx, rows * top * ff, ai.BF16), empty(ai, ctx, rows * top * width, ai.F32), upload(ai, ctx, np.zeros((rows, width)), ai.F32)
    batch = ai.CommandBatch(ctx)
    K.moe_route_into(batch, ai.Buffer.from_slice(ctx, logits), plan, rows, experts, top)
    K.moe_up_into(batch, upload(ai, ctx, x, ai.BF16), ai.BF16, plan, up, hidden, rows, experts, top, width, ff, 3)
    K.moe_down_into(batch, hidden, ai.BF16, plan, down, slots, rb, rows, experts, top, width, ff)
    batch.commit_and_wait()
    words = plan.as_array(np.uint32)
    S = rows * top
    place = words[2 * S:3 * S].reshape(rows, top)
    assert np.array_equal(words[:S].reshape(rows, top), order) and sorted(place.ravel()) == list(range(S))
    by_expert = np.argsort(order.ravel(), kind="stable")
    assert np.array_equal(place.ravel()[by_expert], np.arange(S))       # experts in order, each one's slots in theirs
    close(download(ai, hidden, S * ff, ai.BF16).reshape(S, ff)[place.ravel()].reshape(rows, top, ff), hidden_want, BF16_TOL, "hidden")
    close(download(ai, rb, rows * width, ai.F32).reshape(rows, width), want, BF16_TOL, "sum")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("rows,experts,top,width,ff", [(2, 5, 2, 64, 48), (7, 3, 3, 40, 33), (65, 11, 1, 64, 88), (300, 4, 2, 64, 72), (600, 2, 1, 32, 40),
                                                       (33, 70, 8, 32, 16), (130, 130, 3, 24, 24), (5, 1, 1, 60, 20), (90, 6, 2, 136, 257),
                                                       (3, 300, 4, 24, 16), (2, 4, 3, 4104, 40), (2, 6, 3, 64, 1500)])
def test_mixture_of_experts(ai, gpu, dtype, rows, experts, top, width, ff):
    ctx, K = gpu
    dt = ai.BF16 if dtype == "bf16" else ai.F32
    g = np.random.default_rng(rows + experts)
    x = stored(g.standard_normal((rows, width)), ai, dt)
    ups, downs = (M.rounded(g.standard_normal(s) / np.sqrt(s[2])) for s in ((experts, ff, width), (experts, width, ff)))
    logits = (g.permuted(np.tile(np.arange(experts), (rows, 1)), axis=1) * 0.37 - 1.0).astype(np.float32)
    if experts > 4:
        logits[:, 4] = -50.0                          # an expert that nobody takes
    res = g.standard_normal((rows, width)).astype(np.float32)
    order = np.argsort(-logits, axis=1, kind="stable")[:, :top]
    want, single = res.astype(np.float64), np.zeros((rows, width))
    for t in range(rows):
        for e in order[t]:
            single[t] += downs[e] @ O.relu_squared(ups[e] @ (O.sigmoid(float(logits[t, e])) * x[t]))
    want = want + single
    print(f"experts {dtype} {rows} {experts} {top} {width} {ff}", flush=True)
    plan = ai.Buffer.empty(ctx, 4 * K.moe_plan_words(rows, experts, top))
    up, down = (ai.Buffer.from_slice(ctx, M.bf16_bits(w)) for w in (ups, downs))
    hidden, slots, rb = empty(ai, ctx, rows * top * ff, dt), empty(ai, ctx, rows * top * width, ai.F32), upload(ai, ctx, res, ai.F32)
    lb = ai.Buffer.from_slice(ctx, logits)
    batch = ai.CommandBatch(ctx)
    K.moe_route_into(batch, lb, plan, rows, experts, top)
    K.moe_up_into(batch, upload(ai, ctx, x, dt), dt, plan, up, hidden, rows, experts, top, width, ff, ai.ACT_RELU_SQUARED)
    K.moe_down_into(batch, hidden, dt, plan, down, slots, rb, rows, experts, top, width, ff)
    batch.commit_and_wait()
    assert np.array_equal(plan.as_array(np.uint32, rows * top).reshape(rows, top), order)
    tol = F32_TOL if dt == ai.F32 else BF16_TOL
    close(download(ai, rb, rows * width, ai.F32).reshape(rows, width), want, tol, "residual")
    # one row through the form that selects and norms by itself
    nw, eps = stored(1 + 0.1 * g.standard_normal(width), ai, ai.F32), 1e-5
    h = O.unit_rms(x[0], eps) * nw
    one = sum(downs[e] @ O.relu_squared(ups[e] @ (O.sigmoid(float(logits[0, e])) * h)) for e in order[0])
    rb0, hid = upload(ai, ctx, res[0], ai.F32), empty(ai, ctx, top * ff, ai.F32)
    K.moe_vector_up_into(batch, upload(ai, ctx, x[0], ai.F32), upload(ai, ctx, nw, ai.F32), eps, lb, up, hid, experts, top, width, ff, ai.ACT_RELU_SQUARED)
    K.moe_vector_down_into(batch, hid, lb, down, rb0, experts, top, width, ff)
    batch.commit_and_wait()
    close(download(ai, rb0, width, ai.F32), res[0] + one, F32_TOL, "one row")


@pytest.mark.parametrize("experts,top,width,ff", [(16, 2, 2048, 1024), (8, 2, 1024, 512), (17, 3, 2048, 1024), (5, 5, 512, 40), (32, 4, 1536, 1536), (33, 1, 4096, 900), (1, 1, 64, 8),
                                                  (6, 2, 100, 24), (16, 2, 1368, 688)])
def test_router_in_the_launch_of_the_experts(ai, gpu, experts, top, width, ff):
    """The bits of the router's product and of the experts' own launch behind it, with and without room for the router."""
    ctx, K = gpu
    g = np.random.default_rng(experts * width)
    x, nw = upload(ai, ctx, g.standard_normal(width) * 2, ai.F32), upload(ai, ctx, 1 + 0.1 * g.standard_normal(width), ai.F32)
    router, up = upload(ai, ctx, g.standard_normal((experts, width)) / width ** 0.5, ai.BF16), upload(ai, ctx, g.standard_normal((experts, ff, width)) / width ** 0.5, ai.BF16)
    got = []
    for form in range(2):
        lb, hid, batch = empty(ai, ctx, experts, ai.F32), empty(ai, ctx, top * ff, ai.F32), ai.CommandBatch(ctx)
        if form:
            K.moe_vector_routed_up_into(batch, x, nw, 1e-5, router, lb, up, hid, experts, top, width, ff, ai.ACT_RELU_SQUARED)
        else:
            K.linear_norm_vector_into(batch, x, None, None, nw, 1e-5, router, None, width, ai.linear_weight.Segments([ai.linear_weight.Segment(experts)]), [lb], ai.F32)
            K.moe_vector_up_into(batch, x, nw, 1e-5, lb, up, hid, experts, top, width, ff, ai.ACT_RELU_SQUARED)
        batch.commit_and_wait()
        got.append((lb.as_array(np.uint32), hid.as_array(np.uint32)))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][1].any()


@pytest.mark.parametrize("experts,top,width,ff", [(33, 2, 1536, 256), (64, 4, 2048, 512), (32, 4, 1032, 512), (17, 2, 1024, 512)])
def test_router_beside_the_launch_of_the_experts(ai, gpu, experts, top, width, ff):
    """Around the experts and columns at which the router has a launch of its own and the experts' has four or eight waves."""
    test_router_in_the_launch_of_the_experts(ai, gpu, experts, top, width, ff)


def test_equal_scores_go_to_the_lower_expert(ai, gpu):
    ctx, K = gpu
    logits = np.zeros((3, 9), np.float32)
    logits[1, 6] = logits[1, 2] = 1.0
    plan, batch = ai.Buffer.empty(ctx, 4 * K.moe_plan_words(3, 9, 2)), ai.CommandBatch(ctx)
    K.moe_route_into(batch, ai.Buffer.from_slice(ctx, logits), plan, 3, 9, 2)
    batch.commit_and_wait()
    assert plan.as_array(np.uint32, 6).reshape(3, 2).tolist() == [[0, 1], [2, 6], [0, 1]]
