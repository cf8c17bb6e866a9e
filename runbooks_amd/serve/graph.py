"""hipGraph-captured decode step.

The decode inner loop is launch-bound: ~8 small kernels x num_layers per
step plus five host->device tensor builds. This wraps the whole
model.decode(...) call in a hipGraph (torch.cuda.CUDAGraph is hipGraph on
ROCm) per batch-size bucket: static device input buffers are filled from
pinned staging with async copies, then one graph replay launches the
whole step (graph-replay floor ~10-16 us vs ~3.5 us/launch eager).

Batch sizes are bucketed to powers of two; short batches pad with a
dummy sequence that reads/writes a reserved KV block, so replay shapes
stay fixed while requests come and go.
"""
from __future__ import annotations

import torch

from ..ops.linear import copies_read

RING = 8        # staging buffers


def fixed_nsplit(batch: int, hkv: int, mfma: bool = False) -> int:
    """The most parts of a sequence for the paged-decode kernel, chosen per
    bucket at capture time (paged_decode_parts in csrc/attention_decode.hip
    takes fewer where they would not pay: short tables, or two parts of few
    query heads; the eager heuristic in ops/attention.py reads seq_lens.max() —
    a host sync, impossible inside a graph). base = batch*hkv workgroups
    per split; split until ~4x256 CUs are covered — the head-split GQA
    kernels run 4-5 waves/SIMD, so ~4 WGs/CU (1024 WGs) fills the
    machine (measured sweep: llama2-70b B=32 len-2048 1.75 vs 0.67
    TB/s, falcon MQA 0.72 vs 0.23, B=8 0.99-1.24 vs 0.16 —
    profiles/decode_attn_pipeline.md)."""
    base = max(1, batch * hkv)
    # MFMA path (transposed-V caches): per-wave work is block-granular
    # and latency-light — ~512 WGs is the knee (measured: llama2-70b
    # B=32 len-2048 best at nsplit 2, B=8 at 4-8); the scalar kernels
    # want ~1024.
    target = 512 if mfma else 1024
    if base >= target:
        return 1
    return min(16, max(1, target // base))


class GraphedDecoder:
    def __init__(self, model, caches, max_batch: int, max_blocks: int,
                 dummy_block: int, device, dummy_slot: int = 0):
        self.model = model
        self.caches = caches
        self.device = device
        self.max_blocks = max_blocks
        self.dummy_block = dummy_block
        self.dummy_slot = dummy_slot
        self.buckets = []
        b = 1
        while b < max_batch:
            self.buckets.append(b)
            b *= 2
        self.buckets.append(max_batch)

        B = max_batch
        dev = device
        pin = dict(dtype=torch.int64,
                   pin_memory=torch.cuda.is_available())
        # a step's inputs leave their buffer when the GPU comes to its copy, so
        # steps that are called without waiting need one each: two halves of a
        # ring, an event behind the copies of each (one for every step took 4
        # us of 503)
        self._ring = list(torch.zeros(RING, B * 6 + B * max_blocks, **pin))
        self._sent = [None, None]
        self._turn = -1
        self.h_staging = self._ring[0]
        self._np = self.h_staging.numpy()
        # the same on the device, as it arrives and as the kernels take it
        self.arrived = torch.zeros(self.h_staging.shape, dtype=torch.int64,
                                   device=dev)
        self.inputs = torch.zeros(self.h_staging.shape, dtype=torch.int32,
                                  device=dev)
        # bucket -> (CUDAGraph, logits_out, versions of the weights whose
        # copies it reads)
        self.graphs = {}
        self._pool = None

    # -- capture -----------------------------------------------------------
    def _capture(self, b: int):
        # the runs below must leave live requests alone: a step is not
        # idempotent (recurrent states), and the last step's slots may belong
        # to another request by now
        n = 6 * b + b * self.max_blocks
        for i, value in enumerate((0, 0, self.dummy_block * _bs(), 1, 0,
                                   self.dummy_slot)):
            self.arrived[i * b:(i + 1) * b].fill_(value)
        self.arrived[6 * b:n].fill_(self.dummy_block)
        nsplit = self.model.decode_nsplit(b, self.caches)
        positions, slots, seq_lens, seq_starts, state_slots = \
            self.inputs[b:6 * b].view(5, b)
        tables = self.inputs[6 * b:n].view(b, self.max_blocks)
        args = (self.arrived[:b], positions, self.caches, slots, tables,
                seq_lens)
        kw = dict(nsplit=nsplit, seq_starts=seq_starts)
        if self.model.ragged:
            kw["state_slots"] = state_slots

        def step():
            self.inputs[:n].copy_(self.arrived[:n])
            return self.model.decode(*args, **kw)

        # warmup outside the graph (allocator + autotune settle)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(2):
                step()
        torch.cuda.current_stream().wait_stream(s)

        g = torch.cuda.CUDAGraph()
        with copies_read() as versions:
            if self._pool is None:
                with torch.cuda.graph(g):
                    out = step()
                self._pool = g.pool()
            else:
                with torch.cuda.graph(g, pool=self._pool):
                    out = step()
        self.graphs[b] = (g, out, *versions)

    # -- replay ------------------------------------------------------------
    def decode(self, tokens, positions, slots, block_rows, seq_lens,
               seq_starts=None, state_slots=None):
        """All args host lists; block_rows is a list of per-seq block lists.
        Returns logits [len(tokens), V] (a view into the static output)."""
        n = len(tokens)
        b = next(x for x in self.buckets if x >= n)
        if b not in self.graphs or not self.graphs[b][2].current():
            # not yet, or weights have changed since: their products then run
            # without a copy
            self._capture(b)
        g, out, _ = self.graphs[b]
        self._next_buffer()
        bt = self._stage(b, tokens, positions, slots, block_rows, seq_lens,
                         seq_starts or [0] * n, state_slots)

        # one copy, and one launch within the graph: as seven tensors, each
        # converted on the way, they were 13 launches (a step of opt-125m 533
        # and 511 us)
        size = 6 * b + bt.numel()
        self.arrived[:size].copy_(self.h_staging[:size], non_blocking=True)
        g.replay()
        return out[:n]

    def _next_buffer(self) -> None:
        """Turns to the next staging buffer once its last inputs have left."""
        self._turn = (self._turn + 1) % RING
        half, place = divmod(self._turn, RING // 2)
        if place == 0:
            # every copy of the other half is on its way, also where a step
            # ended early
            self._sent[1 - half] = torch.cuda.Event()
            self._sent[1 - half].record()
            if self._sent[half] is not None:
                self._sent[half].synchronize()
        self.h_staging = self._ring[self._turn]
        self._np = self.h_staging.numpy()

    def _stage(self, b, tokens, positions, slots, block_rows, seq_lens,
               seq_starts, state_slots=None):
        """Fill the pinned staging buffer for bucket size b (numpy view:
        C-speed fills instead of one small torch.tensor per row). Unit-
        tested on CPU (the rest of this class needs a GPU)."""
        n = len(tokens)
        mb = self.max_blocks
        hn = self._np
        hn[0:n] = tokens
        hn[b:b + n] = positions
        hn[2 * b:2 * b + n] = slots
        hn[3 * b:3 * b + n] = seq_lens
        hn[4 * b:4 * b + n] = seq_starts
        hn[5 * b:5 * b + n] = self.dummy_slot if state_slots is None \
            else state_slots
        btn = hn[6 * b:6 * b + b * mb].reshape(b, mb)
        btn.fill(self.dummy_block)
        for i, row in enumerate(block_rows):
            btn[i, :len(row)] = row
        # pad rows beyond n: dummy sequence at position 0, length 1
        if n < b:
            hn[n:b] = 0
            hn[b + n:2 * b] = 0
            hn[2 * b + n:3 * b] = self.dummy_block * _bs()
            hn[3 * b + n:4 * b] = 1
            hn[4 * b + n:5 * b] = 0
            hn[5 * b + n:6 * b] = self.dummy_slot
        return self.h_staging[6 * b:6 * b + b * mb].view(b, mb)


def _bs() -> int:
    from .. import ops
    return ops.BLOCK_SIZE
