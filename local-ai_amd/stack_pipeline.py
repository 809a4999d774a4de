"""Pipeline of a stack of layers with bf16 weights (mixers.py): embedding, layer runs in order -- a range of layers may run
several times in a row -- final norm and head, over the caches and states of sequence slots."""
from __future__ import annotations

from dataclasses import dataclass
from typing import List, Optional, Sequence, Tuple, Type

import numpy as np

from . import BF16, F32, Buffer, CommandBatch, InvalidArgument, Kernels, encoded_work_ran
from .kv_cache import SequenceSlot, SlotPool
from .linear_weight import Segment, StackedLinear
from .mixers import NO_ROW, LatentAttentionSpec, LayerSpec, Norm, OutputNormLayer, PreNormLayer, Run, Workspace

DEFAULT_MAX_ROWS = 2048     # rows of one pass; longer portions go through in pieces


@dataclass
class Loop:
    """The range [start, stop) of layers is walked `times` times; every repetition begins by adding the embedded tokens again."""
    start: int
    stop: int
    times: int


@dataclass
class StackConfig:
    vocab: int
    width: int
    eps: float
    layers: List[LayerSpec]
    loop: Optional[Loop] = None
    layer: Type[PreNormLayer] = PreNormLayer     # where the norms are
    softcap: Optional[float] = None              # logits become softcap * tanh(logits / softcap)

    def runs(self) -> List[Tuple[int, bool]]:
        """[(layer, whether the embedding output is added before it)] in running order."""
        n = len(self.layers)
        if self.loop is None:
            return [(i, False) for i in range(n)]
        a, b, t = self.loop.start, self.loop.stop, self.loop.times
        if not (0 <= a <= b <= n and t >= 0):
            raise InvalidArgument(f"loop over layers {a}..{b} of {n}, {t} times")
        return ([(i, False) for i in range(a)] + [(i, p > 0 and i == a) for p in range(t) for i in range(a, b)]
                + [(i, False) for i in range(b, n)])

    def check(self) -> None:
        """Refuses what no pipeline can run."""
        if self.loop is not None and issubclass(self.layer, OutputNormLayer):
            raise InvalidArgument("layers with norms behind the branches do not repeat")
        if self.softcap is not None and not self.softcap > 0:
            raise InvalidArgument(f"logits capped at {self.softcap}")
        for i, l in enumerate(self.layers):
            m = l.mixer
            if not isinstance(m, LatentAttentionSpec) or m.kv_from is None:
                continue
            j = self.layers[m.kv_from].mixer if 0 <= m.kv_from < i else None
            if not isinstance(j, LatentAttentionSpec) or j.kv_from is not None:
                raise InvalidArgument(f"layer {i} reads the cache of layer {m.kv_from}, which is no earlier layer with one of its own")
            if (j.kv_rank, j.rot_dim, j.rot_base) != (m.kv_rank, m.rot_dim, m.rot_base):
                raise InvalidArgument(f"layer {i} reads the cache of layer {m.kv_from}, whose rows are others")
            if self.loop is not None:
                raise InvalidArgument("layers that share a cache do not repeat")


class StackPipeline:
    """Serves one sequence per slot; the calls are those of generation.SequenceModel."""

    def __init__(self, ctx, kernels: Kernels, config: StackConfig, tensors, max_tokens: int, dtype: int = BF16,
                 max_sequences: int = 1, max_rows: int = DEFAULT_MAX_ROWS, graphs: bool = True):
        if dtype not in (BF16, F32):
            raise InvalidArgument("activations are bf16 or f32")
        config.check()
        self.ctx, self.kernels, self.config, self.dtype, self.graphs = ctx, kernels, config, dtype, graphs
        self.vocab_size, self.max_rows = config.vocab, max_rows
        self.max_tokens = max(max_tokens, 1)
        w = config.width
        self.layers = [config.layer(ctx, kernels, s, w, config.eps, tensors, f"l{i}.") for i, s in enumerate(config.layers)]
        self.runs = config.runs()
        self.embed = Buffer.from_slice(ctx, tensors.bf16("embed", (config.vocab, w)))
        self.final_norm = Norm(ctx, tensors.f32("final.norm", (w,)), config.eps)
        self.head = StackedLinear(ctx, [tensors.bf16("head", (config.vocab, w))], [Segment(config.vocab)])
        self.ws = Workspace(ctx)
        self.tokens_buf = Buffer.empty(ctx, 4 * max_rows)
        self.logits_buf = Buffer.empty(ctx, 4 * config.vocab)
        self.logits_host = Buffer.pinned(ctx, 4 * config.vocab)   # one row, behind a step
        self.next_buf = Buffer.empty(ctx, 4)
        self.at_buf = Buffer.empty(ctx, 4)                # where the token of a step stands
        self.slots = SlotPool(self._new_slot, max_sequences)
        self.observe = None          # called with (run index, residual stream buffer, rows) after every layer run

    def _new_slot(self) -> SequenceSlot:
        memories = []
        for i, _ in self.runs:
            mixer = self.layers[i].mixer
            source = getattr(mixer, "source", None)         # the layer whose memory this one reads
            memories.append(mixer.memory(self.ctx, self.kernels, self.max_tokens, self.dtype) if source is None else memories[source])
        return SequenceSlot(self.ctx, memories)

    # ---- sequences ------------------------------------------------------------------------------------------------------
    def new_sequence(self) -> SequenceSlot:
        return self.slots.acquire()

    def end_sequence(self, seq: SequenceSlot) -> None:
        self.slots.release(seq)

    def step(self, seq: SequenceSlot, tokens: Sequence[int], want: Sequence[int] = ()) -> np.ndarray:
        """Runs `tokens` at the sequence's next positions; logits f32 [len(want), vocab] at those places among them.  All pieces but
        the last are only encoded: if the wait behind them reports a fault, the sequence is where it was."""
        n = len(tokens)
        if n == 0:
            raise InvalidArgument("a step needs at least one token")
        if seq.position + n > self.max_tokens:
            raise InvalidArgument(f"position {seq.position + n} beyond the {self.max_tokens} tokens of a sequence")
        if any(not 0 <= int(t) < self.vocab_size for t in tokens):
            raise InvalidArgument("token id outside the vocabulary")
        if any(not 0 <= int(p) < n for p in want):
            raise InvalidArgument("wanted place outside the step")
        out = np.empty((len(want), self.vocab_size), np.float32)
        begin = seq.position
        try:
            for lo in range(0, n, self.max_rows):
                hi = min(lo + self.max_rows, n)
                at = [i for i, p in enumerate(want) if lo <= p < hi]
                got = out if len(at) == len(want) else np.empty((len(at), self.vocab_size), np.float32)
                self._forward(seq, tokens[lo:hi], [want[i] - lo for i in at], got, wait=hi == n)
                if at and got is not out:
                    out[at] = got
        except BaseException as e:
            if seq.position != begin and not encoded_work_ran(self.ctx, e):
                seq.position = begin
            raise
        return out

    def greedy(self, seq: SequenceSlot, token: int) -> int:
        """One decoded token whose successor is picked on the device."""
        if seq.position + 1 > self.max_tokens:
            raise InvalidArgument(f"position {seq.position + 1} beyond the {self.max_tokens} tokens of a sequence")
        batch = self._decode(seq, token, pick=True)
        picked = int(self.next_buf.as_array(np.uint32, 1)[0])
        self._finish(batch, seq, 1)
        return picked

    # ---- encoding -------------------------------------------------------------------------------------------------------
    def _encode_stack(self, batch, seq: SequenceSlot, n: int, max_position: int, only: Optional[int] = NO_ROW):
        """Embedding and all layer runs of the n tokens in tokens_buf; returns the residual stream: of several tokens that of row `only`,
        where it names one, and nothing to be read where it is NO_ROW; and, of one row, what `_encode_head` has still to add to it.  The embedding output
        stays as it is (later passes of a loop add it): the first norm leaves the stream in a buffer of its own.  For one
        token a norm may not write what other workgroups still read, so the stream alternates between two buffers."""
        x0 = self.ws.get("embedded", n * self.config.width * 4)
        self.kernels.embed_rows_bf16_into(batch, self.embed, self.vocab_size, self.config.width, self.tokens_buf, n, x0)
        return self._encode_layers(batch, seq, n, max_position, x0, seq.position_buf, only if n > 1 and self.observe is None else None)

    def _encode_layers(self, batch, seq: SequenceSlot, n: int, max_position: int, x0: Buffer, position: Buffer, only: Optional[int] = None):
        """With `only` the last layer ends where the rows' keys, values and states are written for all rows but that one: the final norm
        and the head read no other (two passes of 2048 rows, four layers with a routed feed-forward last: 2768 us for all rows, 2501 so)."""
        K, width = self.kernels, self.config.width
        x, y = self.ws.get("stream", n * width * 4), self.ws.get("stream.other", width * 4)
        r = Run(K, batch, n, self.ws, self.dtype, position, max_position, x0, None, x)
        for i, ((layer, add), memory) in enumerate(zip(self.runs, seq.memories)):
            if add:
                r.add = x0
                r.store = (y if r.x is x else x) if n == 1 else r.x
            if i == len(self.runs) - 1:
                r.only = only
            self.layers[layer].run(r, memory)
            if self.observe is not None:
                Norm.flush(r)
                self.observe(i, r.x, n)
        pending = r.pending if r.rows == 1 and self.observe is None else None
        if pending is None:
            Norm.flush(r)
        if only is None or only == NO_ROW or r.rows < n:
            return r.x, pending
        return r.x.view(only * width * 4, width * 4), None

    def _forward(self, seq: SequenceSlot, tokens, want, out: np.ndarray, wait: bool) -> None:
        """Results are read behind the work, in stream order: one wait for both, and for all pieces of a step."""
        n = len(tokens)
        if n == 1 and self.observe is None:
            batch = self._decode(seq, int(tokens[0]), pick=False)
            if want:
                self.logits_host.read_into(out[0])
                out[1:] = out[0]
            return self._finish(batch, seq, 1, wait)
        K, width = self.kernels, self.config.width
        batch = CommandBatch(self.ctx)
        batch.write(self.tokens_buf, np.asarray(tokens, np.uint32))
        only = int(want[0]) if len(want) == 1 and n > 1 and self.observe is None else None
        x = self._encode_stack(batch, seq, n, seq.position, only) if want else self._encode_stack(batch, seq, n, seq.position)
        K.advance_position_into(batch, seq.position_buf, n)
        logits = None
        if len(want) == 1:
            logits = self.logits_host
            row, pending = x
            self._encode_head(batch, row if only is not None else row.view(want[0] * width * 4, width * 4), pending, logits)
        elif want:
            m = len(want)
            index = self.ws.get("want", 4 * self.max_rows)
            batch.write(index, np.asarray(want, np.uint32))
            logits = self.ws.get("logits", m * self.vocab_size * 4)
            size = 4 if self.dtype == F32 else 2
            h = self.ws.get("wanted", m * width * size)
            K.norm_rows_f32_into(batch, x[0], None, self.final_norm.weight, None, index, h, self.dtype, width, m, self.config.eps)
            self.head.rows_into(batch, K, h, self.dtype, m, [logits], F32)
            self._encode_cap(batch, logits, m)
        if want:
            logits.read_into(out)
        self._finish(batch, seq, n, wait)

    def _finish(self, batch, seq: SequenceSlot, n: int, wait: bool = True) -> None:
        if wait:
            batch.commit_and_wait()
        seq.position += n

    def _encode_head(self, batch, row: Buffer, pending: Optional[tuple], copy: Optional[Buffer] = None) -> None:
        norm, eps, cap = self.final_norm.weight, self.config.eps, self.config.softcap
        if pending is not None and copy is not None:
            branch, outer = pending
            return self.kernels.linear_residual_norm_vector_copied_into(batch, row, branch, outer.weight, outer.eps, norm, eps, self.head.weight, self.head.bias,
                                                                        self.head.k, self.vocab_size, self.logits_buf, copy, 0.0 if cap is None else cap)
        if pending is not None:
            branch, outer = pending
            self.kernels.residual_rows_into(batch, row, branch, outer.weight, row, None, F32, outer.dim, 1, outer.eps)
        if copy is not None:
            self.kernels.linear_norm_vector_copied_into(batch, row, norm, eps, self.head.weight, self.head.bias, self.head.k, self.vocab_size,
                                                        self.logits_buf, copy, 0.0 if cap is None else cap)
        elif cap is None:
            self.head.normed_vector_into(batch, self.kernels, row, norm, eps, [self.logits_buf], F32)
        else:
            self.kernels.linear_norm_vector_capped_into(batch, row, norm, eps, self.head.weight, self.head.bias, self.head.k, self.vocab_size,
                                                        self.logits_buf, cap)

    def _encode_cap(self, batch, logits: Buffer, rows: int) -> None:
        if self.config.softcap is not None:
            self.kernels.softcap_f32_into(batch, logits, rows * self.vocab_size, self.config.softcap)

    def _encode_decode(self, batch, seq: SequenceSlot, max_position: int, pick: bool) -> None:
        if pick:
            self._encode_head(batch, *self._encode_stack(batch, seq, 1, max_position))
            self.kernels.argmax_advance_f32_into(batch, self.logits_buf, self.next_buf, self.vocab_size, seq.position_buf, 1)
        else:
            x0 = self.ws.get("embedded", self.config.width * 4)
            self._encode_head(batch, *self._encode_layers(batch, seq, 1, max_position, x0, self.at_buf), self.logits_host)

    def _decode(self, seq: SequenceSlot, token: int, pick: bool) -> CommandBatch:
        """One token, encoded: logits in logits_buf and, where asked, the largest one's index in next_buf.  The first decoded token of a
        slot runs dispatch by dispatch, the next one records the step into a graph that later ones replay as long as the scratch buffers
        stay where they are (everything that changes from step to step is in device memory).  Without the pick a launch ahead of the
        recorded ones brings the token's row and position, by value, and counts the sequence on."""
        batch = CommandBatch(self.ctx)
        if pick:
            batch.write(self.tokens_buf, np.asarray([token], np.uint32))
        else:
            width = self.config.width
            self.kernels.embed_token_bf16_into(batch, self.embed, self.vocab_size, width, token, seq.position,
                                               self.ws.get("embedded", width * 4), self.at_buf, seq.position_buf)
        try:
            self._launch_decode(batch, seq, pick)
        except BaseException:
            if not pick:
                batch.write(seq.position_buf, np.asarray([seq.position], np.uint32))
            raise
        return batch

    def _launch_decode(self, batch, seq: SequenceSlot, pick: bool) -> None:
        graph, version = seq.graphs.get(pick, (None, -1))
        if graph is not None and version == self.ws.version:
            return graph.launch()
        if not (self.graphs and seq.graph_ready):
            self._encode_decode(batch, seq, seq.position, pick)
            seq.graph_ready = True
            return
        seq.graphs.pop(pick, None)
        batch.begin_capture()
        try:
            self._encode_decode(batch, seq, self.max_tokens - 1, pick)
        except BaseException:
            batch.end_capture()
            raise
        graph = batch.end_capture()
        seq.graphs[pick] = graph, self.ws.version
        graph.launch()
