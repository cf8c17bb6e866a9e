"""TP-aware decoder-only transformer covering the llama / falcon / OPT
families the reference platform serves.

One implementation, three family knobs (ModelConfig):
  * norm: RMSNorm (fused gfx950 kernel) or LayerNorm
  * act: SwiGLU (llama), GELU (falcon), ReLU (OPT)
  * pos: RoPE (fused kernel) or learned embeddings (OPT)
  * parallel_residual: falcon's attn+mlp-in-parallel block
  * GQA/MQA via num_kv_heads (llama2-70b 8, falcon-40b 8, falcon-7b 1)
  * layers: models described layer by layer (models/latent.py,
    models/hybrid.py, models/streams.py, models/dual.py)

Forward modes:
  * ``forward(tokens)``             — training, full causal attention
  * ``prefill(...)``                — fills the paged KV cache, returns
                                      last-position logits
  * ``decode(...)``                 — one token per sequence against the
                                      paged cache (gfx950 decode kernel)
  * ``forward_ragged(...)``         — portions of several sequences in one
                                      batch (layer-by-layer models)

TP: attention QKV is column-parallel (head-sharded), the output
projection row-parallel (one xGMI all-reduce); MLP up column / down row
(second all-reduce). KV heads shard when divisible by tp, otherwise the
KV projection is replicated (MQA at tp>1) and each rank keeps a full KV
cache — 288 GB HBM per GPU makes that the right trade on MI355X.
"""
from __future__ import annotations

import math
import os

import torch
from torch import nn

from .. import ops
from ..parallel import (
    ColumnParallelLinear,
    RowParallelLinear,
    comm,
    gather_from_tp,
)
from ..utils.modules import plain, untouched
from . import decode_chain
from .config import LatentAttentionSpec, ModelConfig
from .dual import DualBlock
from .hybrid import SequentialBlock
from .latent import ParallelBlock
from .ragged import RaggedBatch
from .streams import StreamBlock


def _norm_module(cfg: ModelConfig, dtype):
    if cfg.norm == "rmsnorm":
        return ops.RMSNorm(cfg.hidden_size, eps=cfg.norm_eps, dtype=dtype,
                           offset=cfg.norm_offset)
    if cfg.norm == "dyt":
        return ops.DynamicTanh(cfg.hidden_size, dtype=dtype)
    return nn.LayerNorm(cfg.hidden_size, eps=cfg.norm_eps, dtype=dtype)


class Attention(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype, tp: int):
        super().__init__()
        self.cfg = cfg
        self.tp = tp
        self.dh = cfg.head_dim
        assert cfg.num_heads % tp == 0, "num_heads must divide tp"
        self.hq = cfg.num_heads // tp
        self.kv_sharded = cfg.num_kv_heads % tp == 0
        self.hkv = cfg.num_kv_heads // tp if self.kv_sharded else cfg.num_kv_heads
        self.scale = 1.0 / math.sqrt(self.dh)

        q_out = cfg.num_heads * self.dh
        kv_out = cfg.num_kv_heads * self.dh
        # qwen2-style models carry bias on q/k/v but not on o_proj
        in_bias = cfg.attn_bias or cfg.qkv_bias
        self.q_proj = ColumnParallelLinear(cfg.hidden_size, q_out,
                                           bias=in_bias, tp_size=tp, dtype=dtype)
        if self.kv_sharded:
            self.k_proj = ColumnParallelLinear(cfg.hidden_size, kv_out,
                                               bias=in_bias, tp_size=tp,
                                               dtype=dtype, gather_input=False)
            self.v_proj = ColumnParallelLinear(cfg.hidden_size, kv_out,
                                               bias=in_bias, tp_size=tp,
                                               dtype=dtype, gather_input=False)
        else:  # replicate KV (MQA with tp > num_kv_heads)
            self.k_proj = ops.Linear(cfg.hidden_size, kv_out, bias=in_bias,
                                    dtype=dtype)
            self.v_proj = ops.Linear(cfg.hidden_size, kv_out, bias=in_bias,
                                    dtype=dtype)
        self.o_proj = RowParallelLinear(cfg.num_heads * self.dh, cfg.hidden_size,
                                        bias=cfg.attn_bias, tp_size=tp, dtype=dtype)

    def _qkv(self, x, cos, sin, positions):
        # x: [T, hidden] token-major
        T = x.shape[0]
        if getattr(self, "_qkv_w", None) is not None and \
                not torch.is_grad_enabled():
            # fused inference path (fuse_for_inference): one wide GEMM
            # instead of three skinny ones
            qo = self.hq * self.dh
            kvo = self.hkv * self.dh
            y = ops.fast_linear(x, self._qkv_w)
            q = y[:, :qo].contiguous().view(T, self.hq, self.dh)
            k = y[:, qo:qo + kvo].contiguous().view(T, self.hkv, self.dh)
            v = y[:, qo + kvo:].contiguous().view(T, self.hkv, self.dh)
        else:
            q = self.q_proj(x).view(T, self.hq, self.dh)
            k = self.k_proj(x).view(T, self.hkv, self.dh)
            v = self.v_proj(x).view(T, self.hkv, self.dh)
        if self.cfg.pos == "rope":
            q = ops.rope(q, cos, sin, positions)
            k = ops.rope(k, cos, sin, positions)
        return q, k, v

    def forward_train(self, x, cos, sin, positions, B, S):
        group = getattr(self.q_proj, "_group", None)
        if group is not None and self.cfg.pos == "rope" and \
                self.dh in (64, 128) and cos.dtype == torch.float32 and \
                (torch.is_grad_enabled() or
                 getattr(self, "_qkv_w", None) is None):
            y = group.packed(x)     # sibling adapters, q, k and v side by side
            if y is not None:
                o = ops.packed_attention(y, cos, sin, positions, B, S, self.hq,
                                         self.hkv, self.scale)
                return self.o_proj(o.view(B * S, self.hq * self.dh))
        q, k, v = self._qkv(x, cos, sin, positions)
        q = q.view(B, S, self.hq, self.dh)
        k = k.view(B, S, self.hkv, self.dh)
        v = v.view(B, S, self.hkv, self.dh)
        ordered = {"ordered": True} if self.cfg.act == "relu" else {}
        o = ops.causal_attention(q, k, v, scale=self.scale, **ordered)
        return self.o_proj(o.reshape(B * S, self.hq * self.dh))

    def _fused_append(self, x, kc) -> bool:
        """One product for q, k and v, and one kernel for their rotation and
        the cache (csrc/qkv_fused.hip)."""
        return (getattr(self, "_qkv_w", None) is not None and
                not torch.is_grad_enabled() and
                self.cfg.pos == "rope" and ops.use_hip(x) and
                self.dh in (64, 128, 256) and x.dtype == torch.bfloat16 and
                kc.dtype in (torch.bfloat16, torch.uint8))

    def _out(self, o, parts: bool):
        """The output projection; with `parts`, possibly as parts of its sums
        (ops.rows_parts)."""
        if parts and self.o_proj.bias is None:
            y = ops.rows_parts(o, self.o_proj.weight)
            if y is not None:
                return y
        return self.o_proj(o)

    def forward_prefill(self, x, cos, sin, positions, kc, vc, slot_mapping, B,
                        S, parts=False):
        if self._fused_append(x, kc):
            positions = positions.to(torch.int32)
            slot_mapping = slot_mapping.to(torch.int32)
            y = ops.rows_heads(x, self._qkv_w, cos, sin, positions, kc, vc,
                               slot_mapping, self.hq, rows=True)
            if y is None:
                y = ops.wide_linear(x, self._qkv_w)
                ops.ext().qkv_rope_append_(y, cos, sin, positions, kc, vc,
                                           slot_mapping, self.hq)
            o = ops.ext().flash_prefill_qkv(y, B, S, self.hq, self.hkv,
                                            self.dh, self.scale)
            return self._out(o.view(B * S, self.hq * self.dh), parts)
        q, k, v = self._qkv(x, cos, sin, positions)
        ops.kv_append(k, v, kc, vc, slot_mapping)
        q = q.view(B, S, self.hq, self.dh)
        o = ops.flash_prefill(q, k.view(B, S, self.hkv, self.dh),
                              v.view(B, S, self.hkv, self.dh), scale=self.scale)
        return self.o_proj(o.reshape(B * S, self.hq * self.dh))

    def forward_decode(self, x, cos, sin, positions, kc, vc, slot_mapping,
                       block_tables, seq_lens, nsplit=None, slab_ok=False,
                       seq_starts=None, parts=False):
        B = x.shape[0]
        if self._fused_append(x, kc):
            # fused decode hot path: one wide GEMM, then one kernel doing
            # rope(q), rope(k)->cache, v->cache, quantized where the cache is;
            # or one kernel for all of it
            if kc.dtype == torch.uint8:     # whole numbers of any type
                positions = positions.to(torch.int32)
                slot_mapping = slot_mapping.to(torch.int32)
            q = ops.rows_heads(x, self._qkv_w, cos, sin, positions, kc, vc,
                               slot_mapping, self.hq, rows=False)
            if q is None:
                y = ops.wide_linear(x, self._qkv_w)
                q = ops.ext().qkv_rope_append(y, cos, sin, positions, kc, vc,
                                              slot_mapping, self.hq)
        else:
            q, k, v = self._qkv(x, cos, sin, positions)
            ops.kv_append(k, v, kc, vc, slot_mapping)
        o, oswz = ops.paged_decode_with_operand(
            q, kc, vc, block_tables, seq_lens, scale=self.scale,
            nsplit=nsplit, seq_starts=seq_starts)
        o2 = o.reshape(B, self.hq * self.dh)
        if oswz is not None:
            o2._rb_swz = oswz
        if slab_ok and self.tp == 1 and self.o_proj.bias is None:
            out, _ = ops.decode_linear_raw(o2, self.o_proj.weight)
            return out
        return self._out(o2, parts)


class MLP(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype, tp: int):
        super().__init__()
        self.act = cfg.act
        if cfg.act in ("silu_glu", "gelu_glu"):
            self.gate_proj = ColumnParallelLinear(cfg.hidden_size, cfg.intermediate_size,
                                                  bias=cfg.mlp_bias, tp_size=tp, dtype=dtype)
            self.up_proj = ColumnParallelLinear(cfg.hidden_size, cfg.intermediate_size,
                                                bias=cfg.mlp_bias, tp_size=tp, dtype=dtype,
                                                gather_input=False)
        else:
            self.fc1 = ColumnParallelLinear(cfg.hidden_size, cfg.intermediate_size,
                                            bias=cfg.mlp_bias, tp_size=tp, dtype=dtype)
        self.down_proj = RowParallelLinear(cfg.intermediate_size, cfg.hidden_size,
                                           bias=cfg.mlp_bias, tp_size=tp, dtype=dtype)

    def forward(self, x, slab_ok=False, parts=False):
        if self.act in ("silu_glu", "gelu_glu") and \
                getattr(self, "_gateup_w", None) is not None:
            gelu, down = self.act == "gelu_glu", self.down_proj
            if x.dim() == 2 and x.shape[0] <= 32 and down.bias is None and \
                    down.tp == 1 and plain(RowParallelLinear, down):
                y = ops.few_rows_mlp(x, self._gateup_w, down.weight, gelu,
                                     slab_ok)
                if y is not None:
                    return y
            h = ops.rows_glu(x, self._gateup_w, gelu)
            if h is not None:
                y = ops.rows_parts(h, self.down_proj.weight) \
                    if parts and self.down_proj.bias is None else None
                return self.down_proj(h) if y is None else y
        if self.act == "silu_glu":
            if getattr(self, "_gateup_w", None) is not None and \
                    not torch.is_grad_enabled():
                y = ops.wide_linear(x, self._gateup_w)
                if ops.use_hip(y):
                    I = y.shape[-1] // 2
                    if (y.dtype == torch.bfloat16 and I % 16 == 0 and
                            y.numel() // y.shape[-1] <= 32):
                        h, swz = ops.ext().swiglu_packed_dec(y)
                        h._rb_swz = swz
                        if slab_ok and self.down_proj.bias is None:
                            out, _ = ops.decode_linear_raw(
                                h, self.down_proj.weight)
                            return out
                        return self.down_proj(h)
                    return self.down_proj(ops.ext().swiglu_packed(y))
                half = y.shape[-1] // 2
                return self.down_proj(ops.swiglu(
                    y[:, :half].contiguous(), y[:, half:].contiguous()))
            group = getattr(self.gate_proj, "_group", None)
            y = group.packed(x) if group is not None else None
            if y is not None:
                return self.down_proj(ops.swiglu_packed(y))
            return self.down_proj(ops.swiglu(self.gate_proj(x), self.up_proj(x)))
        if self.act == "gelu_glu":
            # gemma GeGLU (tanh approximation); fused gate/up GEMM +
            # csrc geglu_packed epilogue.
            if getattr(self, "_gateup_w", None) is not None and \
                    not torch.is_grad_enabled():
                y = ops.wide_linear(x, self._gateup_w)
                if ops.use_hip(y):
                    I = y.shape[-1] // 2
                    if (y.dtype == torch.bfloat16 and I % 16 == 0 and
                            y.numel() // y.shape[-1] <= 32):
                        h, swz = ops.ext().geglu_packed_dec(y)
                        h._rb_swz = swz
                        if slab_ok and self.down_proj.bias is None:
                            out, _ = ops.decode_linear_raw(
                                h, self.down_proj.weight)
                            return out
                        return self.down_proj(h)
                    return self.down_proj(ops.ext().geglu_packed(y))
                half = y.shape[-1] // 2
                return self.down_proj(
                    torch.nn.functional.gelu(y[:, :half],
                                             approximate="tanh") *
                    y[:, half:])
            return self.down_proj(
                torch.nn.functional.gelu(self.gate_proj(x),
                                         approximate="tanh") * self.up_proj(x))
        h = self.fc1(x)
        if self.act == "gelu":
            h = torch.nn.functional.gelu(h)
        elif self.act == "gelu_tanh":      # gpt2 "gelu_new"
            h = torch.nn.functional.gelu(h, approximate="tanh")
        else:
            h = torch.relu(h)
        return self.down_proj(h)


class Block(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype, tp: int):
        super().__init__()
        self.cfg = cfg
        self.attn = Attention(cfg, dtype, tp)
        self.mlp = MLP(cfg, dtype, tp)
        self.norm1 = _norm_module(cfg, dtype)
        self.norm2 = None if cfg.single_norm else _norm_module(cfg, dtype)

    def forward(self, x, attn_fn):
        """attn_fn(h) runs the right attention mode on normed input."""
        if self.cfg.parallel_residual:
            if self.cfg.single_norm:
                # falcon-7b: one shared ln feeds both branches
                h = self.norm1(x)
                return x + attn_fn(h) + self.mlp(h)
            # falcon-40b: x + attn(ln_attn(x)) + mlp(ln_mlp(x))
            return x + attn_fn(self.norm1(x)) + self.mlp(self.norm2(x))
        x = x + attn_fn(self.norm1(x))
        return x + self.mlp(self.norm2(x))

    def fuses_residual(self) -> bool:
        """The sums of the residual may go into the norms that follow them."""
        return (self.cfg.norm == "rmsnorm" and
                not self.cfg.parallel_residual and not self.cfg.single_norm and
                plain(Block, self) and
                plain(ops.RMSNorm, self.norm1, self.norm2))

    def adds_parts(self) -> bool:
        """Where fuses_residual(): what its sublayers return goes there straight
        from their last product, so that it may come as parts of its sums."""
        attn = self.attn
        return (type(attn) is Attention and attn.tp == 1 and
                untouched(("forward_prefill", "forward_decode",
                           "forward_pending"), attn, self) and
                plain(MLP, self.mlp) and
                plain(RowParallelLinear, attn.o_proj, self.mlp.down_proj))

    def forward_pending(self, x, delta, attn_fn, parts=False):
        """forward() of a residual whose last term is still to be added:
        x + delta -> (x, delta). With `parts`, the new delta may be parts of
        it (ops.rows_parts)."""
        if delta is None:
            h = self.norm1(x)
        else:
            x, h = ops.rmsnorm_res(x, delta, self.norm1.weight,
                                   self.norm1.eps)
        x, h = ops.rmsnorm_res(x, attn_fn(h), self.norm2.weight,
                               self.norm2.eps)
        return x, self.mlp(h, parts=True) if parts else self.mlp(h)

    def forward_decode_fused(self, x_base, delta, attn_fn):
        """Decode hot path (sequential-residual RMSNorm models): the
        residual add is fused into the next norm's kernel
        (rmsnorm_res_fwd_dec), so the layer's residual chain costs zero
        standalone elementwise launches. Returns (new_base, new_delta)
        with the true hidden state = new_base + new_delta (the caller
        folds the final pending delta into norm_f)."""
        ext = ops.ext()
        eps = self.norm1.eps

        def res_norm(base, d, w, e):
            if d.dtype == torch.float32:      # uncombined split-K slab
                return ext.rmsnorm_res_slab_fwd_dec(base, d, w, e)
            return ext.rmsnorm_res_fwd_dec(base, d, w, e)

        if delta is None:
            y1 = self.norm1(x_base)          # attaches _rb_swz itself
            xr1 = x_base
        else:
            xr1, y1, s1 = res_norm(x_base, delta, self.norm1.weight, eps)
            y1._rb_swz = s1
        a = attn_fn(y1)
        xr2, y2, s2 = res_norm(xr1, a, self.norm2.weight, self.norm2.eps)
        y2._rb_swz = s2
        return xr2, self.mlp(y2, slab_ok=True)


class Transformer(nn.Module):
    def __init__(self, cfg: ModelConfig, dtype=torch.bfloat16,
                 tp: int | None = None, device=None):
        super().__init__()
        self.cfg = cfg
        self.tp = tp if tp is not None else comm.world_size()
        self.dtype = dtype
        self.embed = nn.Embedding(cfg.vocab_size, cfg.hidden_size, dtype=dtype)
        if cfg.pos == "learned":
            self.embed_pos = nn.Embedding(cfg.max_seq_len, cfg.hidden_size, dtype=dtype)
        # layer-by-layer models take ragged batches (portions of prompts
        # beside decoded tokens) through forward_ragged
        self.ragged = cfg.layers is not None
        if self.ragged:
            kind = {"streams": StreamBlock, "dual": DualBlock,
                    "shared": ParallelBlock,
                    "sequence": SequentialBlock}[cfg.layout]
            self.blocks = nn.ModuleList(
                kind(cfg, cfg.layers[i], dtype, self.tp) for i in cfg.owners)
            # (layer, loop pass it starts), in the order of execution: a
            # looped layer, or one whose weights another layer uses, runs,
            # and has a cache, every time
            self.runs = cfg.layer_runs
            self._block_of = {i: n for n, i in enumerate(cfg.owners)}
            if cfg.loop is not None:
                self.loop_in = ops.Linear(2 * cfg.hidden_size,
                                          cfg.hidden_size, bias=False,
                                          dtype=dtype)
                if cfg.loop.step:
                    self.loop_step = nn.Parameter(torch.zeros(
                        cfg.loop.times, cfg.hidden_size, dtype=dtype))
        else:
            self.blocks = nn.ModuleList(Block(cfg, dtype, self.tp)
                                        for _ in range(cfg.num_layers))
        self.norm_f = _norm_module(cfg, dtype)
        # vocab-parallel head at TP>1 (untied vocab divisible by tp):
        # each rank's head GEMM shrinks tp-fold; full logits reassemble
        # with one all-gather over xGMI (B x V/tp bf16 per rank, cheap
        # next to the 8x GEMM saving on a 32k-152k vocab).
        self._lm_vocab_parallel = (self.tp > 1 and
                                   cfg.vocab_size % self.tp == 0 and
                                   not cfg.tie_embeddings)
        if self._lm_vocab_parallel:
            self.lm_head = ColumnParallelLinear(
                cfg.hidden_size, cfg.vocab_size, bias=False,
                tp_size=self.tp, dtype=dtype)
        else:
            self.lm_head = ops.Linear(cfg.hidden_size, cfg.vocab_size,
                                      bias=False, dtype=dtype)
        if cfg.tie_embeddings:
            self.lm_head.weight = self.embed.weight
        if self.ragged:
            mixers = [lay.mixer for lay in cfg.layers]
            # windows of the layers that gather long portions' context
            self.windows = sorted({m.window for m in mixers
                                   if isinstance(m, LatentAttentionSpec)},
                                  key=lambda w: (w is None, w))
            # one table per distinct rotation
            distinct = list(dict.fromkeys(m.rotation for m in mixers
                                          if m.rotation is not None))
            self._rope_of = [None if m.rotation is None
                             else distinct.index(m.rotation) for m in mixers]
            for i, (base, dims, *scaling) in enumerate(distinct):
                cos, sin = ops.rope_tables(dims, cfg.max_seq_len, base,
                                           freq_scaling=(*scaling, None)[0])
                self.register_buffer(f"rope_cos_{i}", cos, persistent=False)
                self.register_buffer(f"rope_sin_{i}", sin, persistent=False)
            self._decode_cu = {}
        elif cfg.pos == "rope":
            cos, sin = ops.rope_tables(cfg.head_dim, cfg.max_seq_len, cfg.rope_theta)
            self.register_buffer("rope_cos", cos, persistent=False)
            self.register_buffer("rope_sin", sin, persistent=False)
        else:
            self.rope_cos = self.rope_sin = None
        self.reset_parameters()
        if device is not None:
            self.to(device)

    def block(self, layer: int):
        """The block of a layer with parameters of its own."""
        return self.blocks[self._block_of[layer]]

    def reset_parameters(self):
        for m in self.modules():
            if isinstance(m, (nn.Linear, ColumnParallelLinear, RowParallelLinear)):  # ops.Linear subclasses nn.Linear
                nn.init.normal_(m.weight, std=0.02)
                if getattr(m, "bias", None) is not None:
                    nn.init.zeros_(m.bias)
            elif isinstance(m, nn.Embedding):
                nn.init.normal_(m.weight, std=0.02)

    # -- shared ----------------------------------------------------------------
    def _embed(self, tokens, positions):
        """Token (+learned position) embedding; gemma scales by
        sqrt(hidden) (cfg.embed_scale, 1.0 elsewhere)."""
        x = self.embed(tokens.reshape(-1))
        if self.cfg.embed_scale != 1.0:
            x = x * self.cfg.embed_scale
        if self.cfg.pos == "learned":
            x = x + self.embed_pos(positions.long())
        return x

    # -- training --------------------------------------------------------------
    def forward(self, tokens: torch.Tensor) -> torch.Tensor:
        """tokens [B, S] -> logits [B, S, V] (training / eval, no cache)."""
        if self.ragged:
            raise NotImplementedError(f"{self.cfg.name}: serving only")
        B, S = tokens.shape
        positions = torch.arange(S, device=tokens.device, dtype=torch.int32)
        positions = positions.repeat(B)
        x = self._embed(tokens, positions)
        ckpt = getattr(self, "grad_checkpointing", False) and \
            torch.is_grad_enabled()

        def run(blk, *args):
            if ckpt:
                # recompute this block's activations in backward: peak
                # activation memory drops from O(layers) to O(1) blocks
                # (full fine-tunes of 70B-class models at long seq; LoRA
                # at default shapes fits 288 GB without it)
                return torch.utils.checkpoint.checkpoint(
                    blk, *args, use_reentrant=False)
            return blk(*args)

        def attention(blk, parts):
            return lambda h: blk.attn.forward_train(
                h, self.rope_cos, self.rope_sin, positions, B, S)

        x = self._last_norm(*self._blocks(x, attention, run))
        logits = self.lm_head(x)
        if self._lm_vocab_parallel:
            logits = gather_from_tp(logits)
        return logits.view(B, S, -1)

    def _blocks(self, x, attention, run=lambda blk, *args: blk(*args),
                delta=None, first=0):
        """All blocks, or those from `first` on; attention(block, parts) is its
        attn_fn, which with `parts` may return parts of its sums. x + delta ->
        the residual and what is still to be added to it (None: nothing)."""
        if delta is None and self._sums_in_layer_norms(x):
            dtype, x = x.dtype, x.float()
            for blk in self.blocks:
                h = ops.norm_res32(blk.norm1, x, delta, dtype)
                delta = attention(blk, False)(h)
                h = ops.norm_res32(blk.norm2, x, delta, dtype)
                delta = blk.mlp(h)
            return x, delta
        blocks = list(self.blocks)[first:]
        fuses = [blk.fuses_residual() for blk in blocks]
        # sums of up to 32 rows come whole: without a look at the modules, which
        # takes the host 10 us a block (a prompt of 20 tokens of llama2-7b is
        # bound by the host: 3.5 ms, 0.4 less without)
        many = x.is_cuda and x.shape[0] > 32 and not torch.is_grad_enabled()
        # the norm after the last block may see a part of the rows
        for blk, fused, then in zip(blocks, fuses, fuses[1:] + [False]):
            if fused:
                parts = many and blk.adds_parts()
                x, delta = run(blk.forward_pending, x, delta,
                               attention(blk, parts),
                               *((True,) if parts and then else ()))
            else:
                if delta is not None:
                    x, delta = x + delta, None
                x = run(blk, x, attention(blk, False))
        return x, delta

    def _sums_in_layer_norms(self, x) -> bool:
        """The residual may be kept in fp32 and added to in the kernels of the
        layer norms (results that are not differentiated)."""
        if not (x.is_cuda and x.dtype == torch.bfloat16 and
                not torch.is_grad_enabled() and self.cfg.norm == "layernorm" and
                not self.cfg.parallel_residual and not self.cfg.single_norm and
                x.dim() == 2 and len(self.blocks) > 0):
            return False
        norms = self._layer_norms()
        return (plain(Block, *self.blocks) and plain(nn.LayerNorm, *norms) and
                all(p["weight"] is not None and p["bias"] is not None and
                    p["weight"].dtype == x.dtype
                    for p in (n._parameters for n in norms)))

    def _layer_norms(self):
        # of every pass: without nn.Module's search for attributes
        norms = [m[name] for m in (blk._modules for blk in self.blocks)
                 for name in ("norm1", "norm2")]
        norms.append(self.norm_f)
        return norms

    def _last_norm(self, x, delta):
        if delta is None:
            return self.norm_f(x)
        if x.dtype == torch.float32 and delta.dtype != x.dtype:
            return ops.norm_res32(self.norm_f, x.contiguous(), delta,
                                  delta.dtype)
        if not plain(ops.RMSNorm, self.norm_f):
            return self.norm_f(x + delta)
        return ops.rmsnorm_res(x, delta, self.norm_f.weight,
                               self.norm_f.eps)[1]

    def enable_grad_checkpointing(self, enabled: bool = True) -> None:
        self.grad_checkpointing = enabled

    # -- serving ---------------------------------------------------------------
    @torch.no_grad()
    def prefill(self, tokens, positions, caches, slot_mapping):
        """tokens [B, S]; caches: list of (k_cache, v_cache) per layer.
        Returns last-position logits [B, V]."""
        if self.ragged:
            raise NotImplementedError("prefill through forward_ragged")
        B, S = tokens.shape
        x = self._embed(tokens, positions)
        cache_of = dict(zip(self.blocks, caches))

        def attention(blk, parts):
            kc, vc = cache_of[blk]
            kw = {"parts": True} if parts else {}
            return lambda h: blk.attn.forward_prefill(
                h, self.rope_cos, self.rope_sin, positions, kc, vc,
                slot_mapping, B, S, **kw)

        def attend(attn, y, kc, vc):
            return ops.ext().flash_prefill_qkv(
                y, B, S, attn.hq, attn.hkv, attn.dh, attn.scale).flatten(2) \
                .flatten(0, 1)

        sums = self._few_rows(x, positions, caches, slot_mapping, attend, True,
                              attention)
        x = self._last_norm(*(None if r is None else r.view(B, S, -1)[:, -1]
                              for r in sums))
        logits = self.lm_head(x)
        return gather_from_tp(logits) if self._lm_vocab_parallel else logits

    @torch.no_grad()
    def decode(self, tokens, positions, caches, slot_mapping, block_tables,
               seq_lens, nsplit=None, seq_starts=None, state_slots=None):
        """tokens [B] (one new token per sequence) -> logits [B, V].
        ``nsplit`` is the most parts that decode attention takes a
        sequence in (required under hipGraph capture, serve/graph.py; fewer
        where they would not pay, csrc/attention_decode.hip);
        ``state_slots`` [B] names the
        sequences' state slots (models with recurrent layers)."""
        B = tokens.shape[0]
        if self.ragged:
            if B not in self._decode_cu:
                self._decode_cu[B] = torch.arange(
                    B + 1, dtype=torch.int32, device=tokens.device)
            return self.forward_ragged(RaggedBatch(
                tokens=tokens, positions=positions, slots=slot_mapping,
                cu_q=self._decode_cu[B], seq_lens=seq_lens,
                block_tables=block_tables, state_slots=state_slots,
                seq_of=self._decode_cu[B][:B], rows=None,
                n_seqs=B, n_short=B, t_short=B, max_q=1, max_keys=None),
                caches)
        if self._affine_chain_ready(tokens, positions, caches, slot_mapping):
            logits = self.lm_head(self._decode_affine_chain(
                tokens, positions, caches, slot_mapping, block_tables,
                seq_lens, nsplit, seq_starts))
            return (gather_from_tp(logits) if self._lm_vocab_parallel
                    else logits)
        x = self._embed(tokens.view(B, 1), positions)
        if (ops.use_hip(x) and x.dtype == torch.bfloat16 and B <= 32 and
                self.cfg.norm == "rmsnorm" and
                not self.cfg.parallel_residual and not self.cfg.single_norm
                and self.cfg.hidden_size % 16 == 0 and
                os.environ.get("RB_FUSED_RESID", "1") == "1"):
            # fused residual chain: zero standalone adds in the hot loop
            delta = None
            layers = decode_chain.layers_of(self, Block, Attention, MLP)
            if layers is not None:
                x, delta = decode_chain.run(
                    self, layers, x, positions, caches, slot_mapping,
                    block_tables, seq_lens, nsplit, seq_starts)
            else:
                for blk, (kc, vc) in zip(self.blocks, caches):
                    fn = lambda h, b=blk, kc=kc, vc=vc: b.attn.forward_decode(  # noqa: E731
                        h, self.rope_cos, self.rope_sin, positions, kc, vc,
                        slot_mapping, block_tables, seq_lens, nsplit=nsplit,
                        slab_ok=True, seq_starts=seq_starts)
                    x, delta = blk.forward_decode_fused(x, delta, fn)
            if delta.dtype == torch.float32:
                _, y, swz = ops.ext().rmsnorm_res_slab_fwd_dec(
                    x, delta, self.norm_f.weight, self.norm_f.eps)
            else:
                _, y, swz = ops.ext().rmsnorm_res_fwd_dec(
                    x, delta, self.norm_f.weight, self.norm_f.eps)
            y._rb_swz = swz
            logits = self.lm_head(y)
            return (gather_from_tp(logits) if self._lm_vocab_parallel
                    else logits)
        if ops.use_hip(x) and B <= 32 and self._affine_ready():
            x = self._decode_affine(x, caches, slot_mapping, block_tables,
                                    seq_lens, nsplit, seq_starts)
            logits = self.lm_head(x)
            return (gather_from_tp(logits) if self._lm_vocab_parallel
                    else logits)
        cache_of = dict(zip(self.blocks, caches))

        def attention(blk, parts):
            kc, vc = cache_of[blk]
            kw = {"parts": True} if parts else {}
            return lambda h: blk.attn.forward_decode(
                h, self.rope_cos, self.rope_sin, positions, kc, vc,
                slot_mapping, block_tables, seq_lens, nsplit=nsplit,
                seq_starts=seq_starts, **kw)

        def attend(attn, q, kc, vc):
            return ops.paged_decode_with_operand(
                q, kc, vc, block_tables, seq_lens, scale=attn.scale,
                nsplit=nsplit, seq_starts=seq_starts)[0].flatten(1)

        sums = self._few_rows(x, positions, caches, slot_mapping, attend, False,
                              attention)
        x = self._last_norm(*sums)
        logits = self.lm_head(x)
        return gather_from_tp(logits) if self._lm_vocab_parallel else logits

    def _few_rows(self, x, positions, caches, slots, attend, joint, attention):
        """_blocks(x, attention), as far as it goes by decode_chain.run_rows."""
        delta, first = None, 0
        if (32 < x.shape[0] <= 64 and ops.use_hip(x) and
                x.dtype == torch.bfloat16 and not torch.is_grad_enabled() and
                os.environ.get("RB_FUSED_RESID", "1") == "1"):
            x, delta, first = decode_chain.run_rows(
                self, x, positions, caches, slots, attend, joint, Block,
                Attention, MLP)
        return self._blocks(x, attention, delta=delta, first=first)

    def _affine_ready(self) -> bool:
        """Every block has its products for _decode_affine, of weights that have
        not changed since, and no module that they do the work of would do
        more."""
        return (os.environ.get("RB_FUSED_RESID", "1") == "1" and
                all(getattr(blk, "_affine", None) is not None and
                    _AffineBlock.plain(blk) and
                    blk._affine.current() for blk in self.blocks) and
                plain(nn.LayerNorm, *self._layer_norms()))

    def _affine_chain_ready(self, tokens, positions, caches, slots) -> bool:
        """_affine_ready, and every workgroup of a product can norm the rows
        for itself, and what it reads lies as its kernel takes it (up to 4 rows
        of up to 4096 columns)."""
        B = tokens.shape[0]
        tables = (self.embed, getattr(self, "embed_pos", None))
        return (tokens.is_cuda and tables[1] is not None and
                self.cfg.embed_scale == 1.0 and
                (B > 4 or max(self.cfg.intermediate_size, self.cfg.num_heads *
                              self.cfg.head_dim) <= 4096) and
                getattr(self.blocks[0], "_affine", None) is not None and
                ops.ext().normed_affine_supported(B, self.cfg.hidden_size) and
                tokens.dim() == 1 and tokens.is_contiguous() and
                tokens.dtype == torch.int64 and
                positions.dtype == slots.dtype == torch.int32 and
                positions.is_contiguous() and slots.is_contiguous() and
                positions.numel() == B and
                all(kc.dtype == torch.bfloat16 and kc.is_contiguous() and
                    vc.is_contiguous() for kc, vc in caches) and
                plain(nn.Embedding, *tables) and
                all(t.max_norm is None for t in tables) and
                self._affine_ready() and
                all(p.dtype == torch.bfloat16 and p.is_contiguous() and
                    p.data_ptr() % 16 == 0
                    for p in (*(t.weight for t in tables),
                              *(p for n in self._layer_norms()
                                for p in (n.weight, n.bias)))))

    def _decode_affine_chain(self, tokens, positions, caches, slots,
                             block_tables, seq_lens, nsplit, seq_starts):
        """Decode of layer-norm models with biases (opt, gpt2), of few rows and
        columns: a launch for a product, the norm before it in it
        (csrc/decode_affine.hip), and for attention. Returns the last norm's
        result."""
        ext = ops.ext()
        res = ext.embed_res32(tokens, positions, self.embed.weight,
                              self.embed_pos.weight)
        rows = ext.affine_in_rows(res.shape[0])
        for blk, (kc, vc) in zip(self.blocks, caches):
            attn, products = blk.attn, blk._affine
            q = products.normed(blk.norm1, res, products.qkv_proj,
                                caches=(kc, vc, slots))
            o, swz = ops.paged_decode_with_operand(
                q.view(-1, attn.hq, attn.dh), kc, vc, block_tables, seq_lens,
                scale=attn.scale, nsplit=nsplit, seq_starts=seq_starts)
            products.add(res, o.flatten(1) if rows else swz, products.o_proj)
            h = products.normed(blk.norm2, res, (products.fc1,), products.act,
                                operand=not rows)
            products.add(res, h, products.down_proj)
        return ops.norm_res32(
            self.norm_f, res, None, self.embed.weight.dtype,
            operand=ops.decode_ready(self.lm_head.weight, res.shape[0]))

    def _decode_affine(self, x, caches, slot_mapping, block_tables, seq_lens,
                       nsplit, seq_starts):
        """Decode of layer-norm models with biases (opt, gpt2): nine launches a
        layer, the residual in fp32. Returns the last norm's result."""
        res, delta = x.float(), None
        for blk, (kc, vc) in zip(self.blocks, caches):
            h = ops.norm_res32(blk.norm1, res, delta, x.dtype, operand=True)
            q, k, v = blk._affine.qkv(h._rb_swz, h.shape[0])
            attn = blk.attn
            q = q.view(-1, attn.hq, attn.dh)
            ops.kv_append(k.view(-1, attn.hkv, attn.dh),
                          v.view(-1, attn.hkv, attn.dh), kc, vc, slot_mapping)
            o, swz = ops.paged_decode_with_operand(
                q, kc, vc, block_tables, seq_lens, scale=attn.scale,
                nsplit=nsplit, seq_starts=seq_starts)
            delta = blk._affine.o(swz, h.shape[0])
            h = ops.norm_res32(blk.norm2, res, delta, x.dtype, operand=True)
            delta = blk._affine.mlp(h._rb_swz, h.shape[0])
        return ops.norm_res32(
            self.norm_f, res, delta, x.dtype,
            operand=ops.decode_ready(self.lm_head.weight, res.shape[0]))

    @torch.no_grad()
    def forward_ragged(self, batch: RaggedBatch, caches):
        """One step of a layer-by-layer model: every token of the batch,
        logits [rows, V] fp32 at the wanted ones. The residual stays fp32;
        each layer's output is added by the norm that follows it."""
        x0 = self.embed(batch.tokens)
        x, delta, contexts = x0.to(torch.float32, copy=True), None, {}
        if self.cfg.streams is not None:
            x = (x * self.cfg.embed_scale)[:, None].repeat(
                1, self.cfg.streams, 1)
        for (i, enters), cache in zip(self.runs, caches):
            if enters is not None:
                x, delta = self._enter_pass(x, delta, x0, enters)
            r = self._rope_of[i]
            rope = None if r is None else (getattr(self, f"rope_cos_{r}"),
                                           getattr(self, f"rope_sin_{r}"))
            delta = self.block(i).step(x, delta, batch, cache, rope, contexts)
        if self.cfg.streams is not None:
            return self._head_of_streams(x, delta, batch.rows)
        if batch.rows is not None:
            x = x.index_select(0, batch.rows)
            delta = delta.index_select(delta.dim() - 2, batch.rows)
        w, n = self.lm_head.weight, x.shape[0]
        ready = ops.decode_ready(w, n)
        y = ops.norm_res32(self.norm_f, x, delta, self.dtype, operand=ready)
        if self.cfg.logit_softcap is not None:
            logits = ops.softcap(
                ops.decode_linear_raw(y, w, f32=True)[0] if ready
                else ops.linear_f32(y, w), self.cfg.logit_softcap)
        else:
            logits = (ops.fast_linear(y, w).float() if ready
                      else ops.linear_f32(y, w))
        return gather_from_tp(logits) if self._lm_vocab_parallel else logits

    def _head_of_streams(self, x, pending, rows):
        """Logits of the streams' sum."""
        if rows is not None:
            x, pending = x.index_select(0, rows), pending.rows(rows)
        w, D = self.lm_head.weight, self.cfg.hidden_size
        ready = D % 32 == 0 and ops.decode_ready(w, x.shape[0])
        y = ops.streams_norm(x, pending, self._all_streams, self._norm_f_v,
                             self.dtype, operand=ready)
        logits = (ops.fast_linear(y, w).float() if ready else
                  ops.linear_f32(y[:, :D], w))
        return gather_from_tp(logits) if self._lm_vocab_parallel else logits

    def fuse_streams(self) -> None:
        """What _head_of_streams reads, from the loaded parameters."""
        self._norm_f_v = self.norm_f.packed()
        self._all_streams = torch.ones(self.cfg.streams,
                                       device=self._norm_f_v.device)

    def _enter_pass(self, x, delta, x0, t: int):
        """The residual loop pass t starts from: one product of the residual
        and the embedding output, plus the pass's vector where there is one.
        Returns (x, pending part of it)."""
        w = self.loop_in.weight
        ready = ops.decode_ready(w, x.shape[0])
        h = ops.join_res32(x, delta, x0, operand=ready)
        if ready:
            slab = ops.decode_linear_raw(h, w, f32=True)[0]
            x, delta = slab[0], slab[1:] if len(slab) > 1 else None
        else:
            x, delta = ops.linear_f32(h, w), None
        if self.cfg.loop.step:
            x += self.loop_step[t]
        return x, delta

    # -- cache helpers ----------------------------------------------------------
    def local_kv_heads(self) -> int:
        return self.blocks[0].attn.hkv

    def kv_bytes_per_block(self, fp8: bool = False) -> int:
        """Cache bytes of one block over all layers."""
        if self.ragged:
            return max(1, sum(self.block(i).block_elements()
                              for i, _ in self.runs) *
                       self.embed.weight.element_size())
        elem = self.cfg.head_dim + 16 if fp8 else self.cfg.head_dim * 2
        return 2 * self.cfg.num_layers * self.local_kv_heads() * \
            ops.BLOCK_SIZE * elem

    def state_bytes(self) -> int:
        """Bytes of one sequence's recurrent states (0: the model has
        none)."""
        if not self.ragged:
            return 0
        return sum(self.block(i).state_bytes() for i, _ in self.runs)

    def decode_nsplit(self, batch: int, caches) -> int | None:
        """Work split of the paged-decode kernel for a captured batch (None
        where the model's own kernels choose it)."""
        if self.ragged:
            return None
        from ..ops.attention import _is_vt
        from ..serve.graph import fixed_nsplit
        return fixed_nsplit(batch, self.local_kv_heads(),
                            mfma=_is_vt(*caches[0][:2]))

    def check_serving(self, device, fp8: bool) -> None:
        """Raise when the serving kernels do not cover this model."""
        if self.ragged:
            if fp8:
                raise NotImplementedError(
                    f"{self.cfg.name}: no fp8 cache for layer-by-layer "
                    f"models")
            for i, blk in zip(self.cfg.owners, self.blocks):
                if torch.device(device).type == "cuda" and not blk.covered():
                    raise NotImplementedError(
                        f"{self.cfg.name}: no kernel for the sizes of layer "
                        f"{i}: {blk.spec}")
        elif torch.device(device).type == "cuda" and \
                self.cfg.head_dim not in (64, 128, 256):
            raise NotImplementedError(
                f"paged decode supports head_dim 64/128/256 on gfx950; "
                f"{self.cfg.name} has {self.cfg.head_dim}")

    def alloc_caches(self, num_blocks: int, device, fp8: bool = False,
                     num_slots: int = 1):
        if self.ragged:
            # one per layer run; a layer that reads another's latents shares
            # its cache
            caches = []
            for i, _ in self.runs:
                src = getattr(self.cfg.layers[i].mixer, "kv_from", None)
                caches.append(caches[src] if src is not None else
                              self.block(i).alloc_cache(num_blocks, num_slots,
                                                        device))
            return caches
        # Transposed-V blocks feed the MFMA decode kernel's direct V^T
        # fragment reads (GQA/MQA models, bf16, Dh<=128). The cache
        # shape is the routing signal all the way down (kv_append,
        # paged_decode). RB_DECODE_MFMA=0 reverts to the scalar path.
        attn = self.blocks[0].attn
        vt = ((fp8 or self.dtype == torch.bfloat16)
              and attn.hq // attn.hkv >= 4 and self.cfg.head_dim <= 128
              and ops.BLOCK_SIZE == 16
              and os.environ.get("RB_DECODE_MFMA", "1") != "0")
        return [ops.alloc_kv_cache(num_blocks, self.local_kv_heads(),
                                   self.cfg.head_dim, device,
                                   dtype=self.dtype, fp8=fp8,
                                   v_transposed=vt)
                for _ in range(self.cfg.num_layers)]


class _AffineBlock:
    """A block's products with their biases and activation in a launch each
    (csrc/decode_affine.hip). They read the parameters, so a
    captured step follows weights that change in place."""

    ACTS = {"relu": 1, "gelu": 2, "gelu_tanh": 3}

    @staticmethod
    def serves(model, blk) -> bool:
        cfg, a, m = model.cfg, blk.attn, blk.mlp
        return (cfg.norm == "layernorm" and cfg.pos == "learned" and
                cfg.act in _AffineBlock.ACTS and not cfg.parallel_residual and
                not cfg.single_norm and model.tp == 1 and
                cfg.hidden_size % 32 == 0 and cfg.hidden_size <= 16384 and
                m.fc1.weight.shape[0] % 32 == 0 and
                a.hq * a.dh % 32 == 0 and a.hkv * a.dh % 32 == 0 and
                all(n.weight is not None and n.bias is not None
                    for n in (blk.norm1, blk.norm2, model.norm_f)) and
                all(t.dtype == torch.bfloat16 and t.is_contiguous() and
                    t.data_ptr() % 16 == 0
                    for p in (a.q_proj, a.k_proj, a.v_proj, a.o_proj, m.fc1,
                              m.down_proj)
                    for t in (p.weight, p.bias) if t is not None))

    @staticmethod
    def plain(blk) -> bool:
        a, m = blk.attn, blk.mlp
        return (plain(Block, blk) and plain(MLP, m) and
                plain(ColumnParallelLinear, a.q_proj, a.k_proj, a.v_proj,
                      m.fc1) and
                plain(RowParallelLinear, a.o_proj, m.down_proj))

    def __init__(self, blk, act: str):
        a, m = blk.attn, blk.mlp
        self.act = self.ACTS[act]
        self.qkv_proj = (a.q_proj, a.k_proj, a.v_proj)
        self.o_proj, self.fc1, self.down_proj = a.o_proj, m.fc1, m.down_proj
        self.sources = [t for p in (*self.qkv_proj, a.o_proj, m.fc1,
                                    m.down_proj)
                        for t in (p.weight, p.bias) if t is not None]
        self.versions = self._versions()

    def _versions(self):
        return [(t.data_ptr(), t.dtype,
                 None if t.is_inference() else t._version)
                for t in self.sources]

    def current(self) -> bool:
        """The parameters are those of the time of fusing."""
        return self._versions() == self.versions

    @staticmethod
    def _products(projections, swz, rows: int, act: int = 0, operand=False):
        return ops.ext().decode_affine(
            swz, [p.weight for p in projections],
            [p.bias for p in projections], rows, act, operand)

    @staticmethod
    def normed(norm, res, projections, act: int = 0, operand=False,
               caches=(None, None, None)):
        """The first product of the norm of a residual; with caches the others
        go there."""
        return ops.ext().normed_affine(
            res, norm.weight, norm.bias, norm.eps,
            [p.weight for p in projections], [p.bias for p in projections],
            act, operand, *caches)[0]

    @staticmethod
    def add(res, x, projection):
        """res += the product."""
        ops.ext().affine_add_(x, projection.weight, projection.bias, res)

    def qkv(self, swz, rows: int):
        return self._products(self.qkv_proj, swz, rows)

    def o(self, swz, rows: int):
        return self._products((self.o_proj,), swz, rows)[0]

    def mlp(self, swz, rows: int):
        h = self._products((self.fc1,), swz, rows, self.act, True)[0]
        return self._products((self.down_proj,), h, rows)[0]


def _fuse_projections(model: "Transformer") -> dict[torch.Tensor, int]:
    """Fused qkv and gate/up weights; returns every layer's serving weights
    with the distance of the rows that their copies pair (0: none)."""
    for blk in model.blocks:
        attn = blk.attn
        if (attn.q_proj.bias is None and
                getattr(attn.k_proj, "bias", None) is None and
                attn.q_proj.weight.shape[1] == attn.k_proj.weight.shape[1]):
            fused = torch.cat([attn.q_proj.weight.data,
                               attn.k_proj.weight.data,
                               attn.v_proj.weight.data], dim=0).contiguous()
            qo = attn.q_proj.weight.shape[0]
            kvo = attn.k_proj.weight.shape[0]
            attn._qkv_w = fused
            attn.q_proj.weight = nn.Parameter(fused[:qo],
                                              requires_grad=False)
            attn.k_proj.weight = nn.Parameter(fused[qo:qo + kvo],
                                              requires_grad=False)
            attn.v_proj.weight = nn.Parameter(fused[qo + kvo:],
                                              requires_grad=False)
        mlp = blk.mlp
        # geglu_packed is default-on, RB_FUSED_GEGLU=0 reverts to eager
        glu_fusable = model.cfg.act == "silu_glu" or (
            model.cfg.act == "gelu_glu" and
            os.environ.get("RB_FUSED_GEGLU", "1") == "1")
        if glu_fusable and mlp.gate_proj.bias is None:
            fused = torch.cat([mlp.gate_proj.weight.data,
                               mlp.up_proj.weight.data],
                              dim=0).contiguous()
            half = mlp.gate_proj.weight.shape[0]
            mlp._gateup_w = fused
            mlp.gate_proj.weight = nn.Parameter(fused[:half],
                                                requires_grad=False)
            mlp.up_proj.weight = nn.Parameter(fused[half:],
                                              requires_grad=False)
    # the copies of weights whose rows meet in what follows the product are
    # paired: a rotation's halves, gate and unit
    def half_of(w, half):
        return half if half % 16 == 0 and w is not None and \
            w.shape[0] % (2 * half) == 0 else 0

    halves = {}
    for blk in model.blocks:
        qkv = getattr(blk.attn, "_qkv_w", None)
        if qkv is not None and model.cfg.pos == "rope":
            halves[qkv] = half_of(qkv, blk.attn.dh // 2)
        gateup = getattr(blk.mlp, "_gateup_w", None)
        if gateup is not None:
            halves[gateup] = half_of(gateup, gateup.shape[0] // 2)
    return {w: halves.get(w, 0) for blk in model.blocks
            for w in (getattr(blk.attn, "_qkv_w", None),
                      getattr(blk.mlp, "_gateup_w", None),
                      blk.attn.o_proj.weight, blk.mlp.down_proj.weight)
            if w is not None}


def fuse_for_inference(model: "Transformer",
                       load_in_8bit: bool = False) -> "Transformer":
    """Fuse each block's QKV and gate/up weights into single tensors for
    serving: one wide GEMM per group instead of 2-3 skinny ones (the
    batch-<=32 decode GEMMs are weight-bandwidth bound, and hipBLASLt is
    markedly more efficient at the fused N — profiles/). The original
    parameters become views into the fused tensor, so no extra HBM and
    the separate-projection training path keeps working.
    """
    if model.ragged:
        weights = {w: 0 for blk in model.blocks for w in blk.fuse()}
        if model.cfg.loop is not None:
            weights[model.loop_in.weight] = 0
        if model.cfg.streams is not None:
            model.fuse_streams()
    else:
        weights = _fuse_projections(model)
    if not load_in_8bit and torch.cuda.is_available() and ops.has_hip() and \
            os.environ.get("RB_DECODE_GEMM", "1") == "1" and \
            model.dtype == torch.bfloat16:
        # Register fragment-lane-major weight copies for the v2 decode
        # GEMM (csrc/decode_gemm.hip): doubles decode-weight memory, which
        # 288 GB HBM3E affords for every served model at TP=1 except
        # llama2-70b (which serves via MODEL_LOAD_IN_8BIT / TP>1). Budget
        # guard: keep at least ~35% of the GPU free for KV cache.
        from ..ops.linear import register_decode_weight
        ext = ops.ext()
        cands = [w for w in weights
                 if ext.decode_gemm_supported(32, w.shape[0], w.shape[1])]
        if model.lm_head.weight.shape[0] % 32 == 0 and \
                ext.decode_gemm_supported(32, model.lm_head.weight.shape[0],
                                          model.lm_head.weight.shape[1]):
            cands.append(model.lm_head.weight)
        need = sum(2 * w.numel() for w in cands)
        free, total = torch.cuda.mem_get_info()
        if free - need >= int(0.35 * total):
            for w in cands:
                register_decode_weight(w, weights.get(w, 0))
        for blk in () if model.ragged else model.blocks:
            if model.lm_head.weight.is_cuda and _AffineBlock.serves(model, blk):
                blk._affine = _AffineBlock(blk, model.cfg.act)

    if load_in_8bit and torch.cuda.is_available():
        # MODEL_LOAD_IN_8BIT: decode weights additionally stored as OCP
        # e4m3 + per-channel scales — the decode GEMM streams half the
        # bytes (ops/csrc/decode_gemm.hip, decode_gemm_fp8). bf16 masters
        # stay for prefill/big-M GEMMs: 288 GB HBM3E makes both-copies the
        # right trade on MI355X.
        from ..ops.linear import quantize_fp8
        for w, half in weights.items():
            if w.shape[0] % 64 == 0 and w.shape[1] % 256 == 0:
                quantize_fp8(w, half)
        if model.lm_head.weight.shape[0] % 64 == 0 and \
                model.lm_head.weight.shape[1] % 256 == 0:
            quantize_fp8(model.lm_head.weight)
    return model


def build_model(name_or_cfg, dtype=torch.bfloat16, tp: int | None = None,
                device=None, seed: int = 0) -> Transformer:
    from .config import get_config
    cfg = name_or_cfg if isinstance(name_or_cfg, ModelConfig) else get_config(name_or_cfg)
    torch.manual_seed(seed)
    if device is not None:
        # construct directly on the target device — a 7B bf16 random init
        # takes minutes on CPU but is instant on the GPU, and 8 DP ranks
        # would otherwise all churn host RAM at once
        with torch.device(device):
            return Transformer(cfg, dtype=dtype, tp=tp)
    return Transformer(cfg, dtype=dtype, tp=tp)
