"""Decode of RMSNorm models of up to 32 sequences, a layer in six launches
(csrc/decode_ends.h, csrc/decode_res.hip):

  * q, k and v, rotated and cached;
  * attention, and the sum of its parts where sequences are split;
  * the output projection with the residual and the next norm's sums;
  * gate and up projection with the gated unit;
  * the down projection with the residual and the next norm's sums.

A norm's 1 / rms is left to the product that reads its result. Long sums and wide
residuals go in parts, with a launch that adds them up (_in_parts). Where a step has
no kernel of either kind (8-bit caches and weights with such sums) it is the launches
of Block.forward_decode_fused.

33 to 64 rows, sequences or tokens of a prompt, go the same way with rows in place
of operands (run_rows).
"""
from __future__ import annotations

import torch

from .. import ops
from ..parallel import ColumnParallelLinear, RowParallelLinear
from ..utils.modules import plain, untouched


class _Layer:
    """Copies that a block's products read."""

    def __init__(self, blk):
        a, m = blk.attn, blk.mlp
        self.blk, self.attn = blk, a
        self.gelu = m.act == "gelu_glu"
        self.qkv, self.o = ops.Copy(a._qkv_w), ops.Copy(a.o_proj.weight)
        self.gate_up = ops.Copy(m._gateup_w)
        self.down = ops.Copy(m.down_proj.weight)

    def served(self) -> bool:
        return (all(c.ws is not None for c in (self.qkv, self.o, self.gate_up,
                                               self.down)) and
                self.qkv.half * 2 == self.attn.dh and
                self.gate_up.half * 2 == self.gate_up.n)


def _served(model) -> bool:
    cfg = model.cfg
    return (cfg.pos == "rope" and cfg.act in ("silu_glu", "gelu_glu") and
            model.tp == 1 and model.rope_cos.dtype == torch.float32)


def _layers(blocks, steps, block_type, attention_type, mlp_type):
    """A _Layer for each of `blocks`, or None where one is not served or a module
    would do more than its kernels (or has `steps` of its own)."""
    mlps, attns = [b.mlp for b in blocks], [b.attn for b in blocks]
    if not (blocks and plain(block_type, *blocks) and plain(mlp_type, *mlps) and
            plain(attention_type, *attns) and
            untouched(steps, *attns, *blocks) and
            plain(ops.RMSNorm, *(n for b in blocks
                                 for n in (b.norm1, b.norm2))) and
            plain(RowParallelLinear, *(m.down_proj for m in mlps),
                  *(a.o_proj for a in attns)) and
            plain(ColumnParallelLinear, *(m.gate_proj for m in mlps),
                  *(m.up_proj for m in mlps), *(a.q_proj for a in attns))):
        return None
    for b in blocks:
        if (getattr(b.attn, "_qkv_w", None) is None or
                getattr(b.mlp, "_gateup_w", None) is None or
                b.attn.o_proj.bias is not None or
                b.mlp.down_proj.bias is not None or
                any(n.weight.dtype != torch.bfloat16 or
                    not n.weight.is_contiguous()
                    for n in (b.norm1, b.norm2))):
            return None
    layers = [_Layer(b) for b in blocks]
    return layers if all(layer.served() for layer in layers) else None


def layers_of(model, *types):
    """A _Layer for every block of a step, or None."""
    return _layers(list(model.blocks),
                   ("forward_decode", "forward_decode_fused"), *types) \
        if _served(model) else None


class _Normed:
    """A norm's result for the products that read it: an operand, rows, or both,
    without its 1 / rms where there are squares."""

    def __init__(self, swz=None, rows=None, squares=None, eps=0.0):
        self.swz, self.rows = swz, rows
        self.squares, self.eps = squares, eps


def _heads(layer, y, m, cos, sin, positions, kc, vc, slots):
    ext, c, hq = ops.ext(), layer.qkv, layer.attn.hq
    if kc.dtype != torch.bfloat16:          # rows of it share a scale
        if y.squares is not None:
            out = ext.decode_normed(y.swz, c.ws, c.scale, m, c.n, c.k,
                                    y.squares, y.eps, c.half)
        else:
            out = ops.wide_linear(y.rows, layer.attn._qkv_w)
        return ext.qkv_rope_append(out, cos, sin, positions.to(torch.int32),
                                   kc, vc, slots.to(torch.int32), hq)
    if y.swz is None or (y.squares is None and c.shares_x(m)):
        return ext.rows_heads(y.rows, c.ws, c.n, cos, sin, positions, kc, vc,
                              slots, hq, False, y.squares, y.eps)
    return ext.decode_heads(y.swz, c.ws, c.scale, m, c.n, c.k, y.squares, y.eps,
                            cos, sin, positions, kc, vc, slots, hq)


def _gate_shares_x(c, m: int) -> bool:
    """shares_x of a gated unit, which the kernel whose waves share x also wins where it
    is wider: of more than 24 rows, unless rows of x begin a multiple of 2 kB apart (few of
    L2's channels have them all) and there is not much of W; of fewer with long sums. us
    by operands and by rows, of 24 and of 32 rows:
      36864 x 3072  39.1 42.0  42.4 43.2    36864 x 3328  45.8 45.9  50.4 47.4
      40960 x 3072  40.6 43.5  44.0 44.4    33792 x 3584  46.2 47.9  51.1 49.3
      49152 x 3072  48.0 47.1  52.2 47.9    40960 x 3584  49.0 50.0  53.9 51.3
      57344 x 3072  55.6 55.6  60.8 56.0    40960 x 3840  51.6 53.2  56.2 55.1
      36864 x 4096  51.9 59.7  56.4 60.5    36864 x 4352  58.0 58.3  63.6 60.4
      43008 x 4096  60.7 61.6  66.4 62.7    40960 x 4608  61.4 63.0  67.3 64.6
      49152 x 4096  63.8 67.8  69.0 69.1    36864 x 5632  71.2 73.9  78.5 75.8
      57344 x 4096  74.1 74.5  80.4 74.9    33792 x 6656  81.5 85.0  89.9 87.0
      40960 x 5120  65.1 70.2  70.7 73.1    40960 x 6656  86.8 89.0  95.0 91.5
      43008 x 5120  74.2 71.4  81.5 73.8    36864 x 6144  74.4 80.3  81.6 82.9
      57344 x 5120  90.5 88.6  98.6 89.6    44032 x 8192 120.8 113.0 130.9 114.3
    and of 65536 x 4096 83.7 and 84.6, 90.5 and 84.5. Results in rows take the kernel
    for operands 0.5 to 7 us more."""
    wide = 16 < m <= 32 and not c.fp8 and 32768 < c.n <= 57344
    if m <= 24:
        return c.shares_x(m) or (wide and c.n >= 43008 and c.k >= 5120)
    return c.shares_x(m) or (wide and c.k >= 3072 and
                             (c.n >= 43008 or c.k % 1024 != 0))


def _gated(layer, y, m, operand: bool):
    ext, c = ops.ext(), layer.gate_up
    if y.rows is not None and (y.swz is None or _gate_shares_x(c, m)):
        return ext.rows_glu(y.rows, c.ws, c.n, layer.gelu, operand, y.squares,
                            y.eps)
    return ext.decode_glu(y.swz, c.ws, c.scale, m, c.n, c.k, layer.gelu,
                          y.squares, y.eps, not operand)


def _add(x, operand, copy, norm, rows: bool):
    """x + operand W^T and its norm, as rows where those will do."""
    ext, m = ops.ext(), x.shape[0]
    # the kernel whose workgroups have whole sums reads x once for 16 columns,
    # which is what it takes with many long rows (us in parts and whole, with
    # the norm: 32 rows, 4096 x 4096 13.8 and 10.3, 4096 x 11008 25.2 and 25.1,
    # 4096 x 14336 29.7 and 33.5, 3072 x 24576 42.1 and 49.5; 16 rows 12.7 and
    # 8.5, 22.3 and 21.0, 25.4 and 24.1, 37.2 and 37.6); long ones are _in_parts'
    if (m <= 16 or copy.k <= 8192) and \
            ext.decode_res_supported(m, copy.n, copy.k, copy.fp8):
        x, y, squares = ext.decode_res(operand, copy.ws, copy.scale, x,
                                       norm.weight, rows)
        return x, _Normed(None if rows else y, y if rows else None, squares,
                          norm.eps)
    delta = copy.product(operand, m)
    add = (ext.rmsnorm_res_slab_fwd_dec if delta.dtype == torch.float32 else
           ext.rmsnorm_res_fwd_dec)
    x, rows_, swz = add(x, delta, norm.weight, norm.eps)
    return x, _Normed(swz, rows_)


def _in_parts(copy, m: int) -> bool:
    """Whether the sums of up to 32 rows that get the residual go as those of 33 to 64
    do: in parts by the kernel whose waves share x, and a launch that adds them up
    (_add_rows). us of the product and the norm by operands in parts, so, and in whole
    sums, weights out of cache, of 1, 16, 17 and 32 rows:
      3072 x 24576  33.6 27.8 30.8  34.3 27.5 32.8  35.3 27.6 38.6  38.7 29.4 45.0
      4096 x 11008  20.2 18.6 18.6  21.3 18.4 19.4  21.8 18.4 20.7  23.7 19.9 23.8
      4096 x 8192   19.2 16.4 13.6  20.0 16.6 13.9  20.0 16.7 15.8  20.3 17.1 17.9
      5120 x 5120   16.7 13.0       18.2 14.0       19.6 14.1       21.6 15.6
      5120 x 13824  33.5 28.7       35.8 31.1       37.6 29.0       42.0 32.1
    Of up to 16 rows what the products around it lose by rows (0 to 0.7 us) is more
    than 4096 x 11008 gains."""
    ext = ops.ext()
    return (not copy.fp8 and copy.half == 0 and copy.n <= 8192 and
            ext.parts_res_supported(copy.n) and copy.k >= 1024 and
            (copy.k > (16384 if m <= 16 else 8192) or
             not ext.decode_res_supported(m, copy.n, copy.k, False)))


def _heads_by_rows(layer, m: int, kc) -> bool:
    c = layer.qkv
    return (not c.fp8 and c.k >= 1024 and kc.dtype == torch.bfloat16 and
            layer.blk.norm1.weight.data_ptr() % 16 == 0 and
            ops.ext().rows_ends_pay(m, c.n, c.k))


def _gate_by_rows(layer, m: int) -> bool:
    """us by operands and by rows, of 1, 8 and 16 rows: 27648 x 5120 48.0 44.1, 45.8
    43.8, 46.3 44.3; 28672 x 4096 40.1 41.1, 39.2 38.9, 39.4 39.6; 49152 x 3072 47.0
    52.4, 45.1 50.9, 44.6 51.5."""
    c = layer.gate_up
    return (not c.fp8 and c.k >= 1024 and 10240 <= c.n <= 32768 and
            layer.blk.norm2.weight.data_ptr() % 16 == 0)


def run(model, layers, x, positions, caches, slots, tables, seq_lens, nsplit,
        seq_starts):
    """x [m, hidden], embedded tokens -> (residual, what the last block has
    still to add to it: bf16 [m, hidden] or fp32 parts of it)."""
    ext, m = ops.ext(), x.shape[0]
    cos, sin = model.rope_cos, model.rope_sin
    norm = layers[0].blk.norm1
    rows, swz = ext.rmsnorm_fwd_dec(x, norm.weight, norm.eps)
    y = _Normed(swz, rows)
    for i, (layer, (kc, vc)) in enumerate(zip(layers, caches)):
        blk, attn = layer.blk, layer.attn
        q = _heads(layer, y, m, cos, sin, positions, kc, vc, slots)
        o, operand = ops.paged_decode_with_operand(
            q, kc, vc, tables, seq_lens, scale=attn.scale, nsplit=nsplit,
            seq_starts=seq_starts)
        if _in_parts(layer.o, m) and _gate_by_rows(layer, m):
            x, y = _add_rows(x, o.view(m, -1), layer.o, blk.norm2)
        else:
            x, y = _add(x, operand, layer.o, blk.norm2,
                        _gate_shares_x(layer.gate_up, m))
        after = layers[i + 1] if i + 1 < len(layers) else None
        rows = (after is not None and _in_parts(layer.down, m) and
                _heads_by_rows(after, m, caches[i + 1][0]))
        h = _gated(layer, y, m, not rows)
        if rows:
            x, y = _add_rows(x, h, layer.down, after.blk.norm1)
        elif after is not None:
            x, y = _add(x, h, layer.down, after.blk.norm1, False)
    return x, layers[-1].down.product(h, m)


def _rows_layer(blk, m: int, kc, types):
    """blk's _Layer where its kernels serve m rows, else None."""
    layers = _layers([blk], ("forward_prefill", "forward_decode",
                             "forward_pending"), *types)
    if layers is None or kc.dtype != torch.bfloat16:
        return None
    y, pays = layers[0], ops.ext().rows_ends_pay
    return y if (not any(c.fp8 for c in (y.qkv, y.o, y.gate_up, y.down)) and
                 min(y.qkv.k, y.o.k, y.down.k) >= 1024 and
                 all(n.weight.data_ptr() % 16 == 0
                     for n in (blk.norm1, blk.norm2)) and
                 pays(m, y.qkv.n, y.qkv.k) and
                 pays(m, y.gate_up.n, y.gate_up.k)) else None


def _add_rows(x, rows, copy, norm):
    """x + rows W^T and its norm: whole sums with the residual behind them, or, of
    long rows, parts and a launch that adds them up (us of 45 and 64 rows, in parts
    with the norm and whole: 4096 x 4096 15.8 and 12.2, 16.4 and 13.5; 2048 x 2048
    11.2 and 7.6, 11.9 and 8.2; 4096 x 11008 26.6 and 28.6, 28.6 and 32.6; 4096 x
    14336 28.8 and 37.6, 30.8 and 39.6). Prompts of 45 tokens of llama2-7b, one after
    the other, take 3457 us in the modules' launches and 3309 in run_rows'."""
    ext, m = ops.ext(), x.shape[0]
    if copy.half == 0 and copy.k <= 8192 and \
            ext.rows_res_supported(m, copy.n, copy.k):
        x, y, squares = ext.rows_res(rows, copy.ws, x, norm.weight)
        return x, _Normed(rows=y, squares=squares, eps=norm.eps)
    delta = ext.decode_gemm_rows(rows, copy.ws, copy.n, copy.half, True)
    if delta.dim() == 3:
        x, y, squares = ext.parts_res(delta, x, norm.weight)
        return x, _Normed(rows=y, squares=squares, eps=norm.eps)
    x, y = ops.rmsnorm_res(x, delta, norm.weight, norm.eps)
    return x, _Normed(rows=y)


def run_rows(model, x, positions, caches, slots, attend, joint: bool, *types):
    """x [m, hidden], 33 to 64 embedded tokens, through the blocks up to the first
    that is not served -> (residual, what the last of them has still to add to it
    or None, how many they are). attend(attention, q, keys, values) returns the
    heads' results as rows; with `joint`, q is q, k and v side by side.

    A block is looked at while the GPU is at the one before it: a look at all of
    llama2-7b takes the host 0.7 ms, for which an idle GPU would wait (a prompt of 45
    tokens by itself, from the call until its logits are there: 4.22 ms, so 3.52, and
    3.70 in the modules)."""
    cfg, ext, m = model.cfg, ops.ext(), x.shape[0]
    if not (_served(model) and cfg.norm == "rmsnorm" and
            not cfg.parallel_residual and not cfg.single_norm and
            cfg.head_dim in (64, 128, 256) and
            ext.parts_res_supported(cfg.hidden_size)):
        return x, None, 0
    blocks = list(model.blocks)
    layer = _rows_layer(blocks[0], m, caches[0][0], types) if blocks else None
    if layer is None:
        return x, None, 0
    cos, sin = model.rope_cos, model.rope_sin
    positions = positions.to(torch.int32)
    slots = slots.to(torch.int32)
    norm = layer.blk.norm1
    y = _Normed(rows=ops.rmsnorm(x, norm.weight, norm.eps))
    for i, (kc, vc) in enumerate(caches, 1):
        c = layer.qkv
        q = ext.rows_heads(y.rows, c.ws, c.n, cos, sin, positions, kc, vc,
                           slots, layer.attn.hq, joint, y.squares, y.eps)
        x, y = _add_rows(x, attend(layer.attn, q, kc, vc), layer.o,
                         layer.blk.norm2)
        c, down = layer.gate_up, layer.down
        h = ext.rows_glu(y.rows, c.ws, c.n, layer.gelu, False, y.squares, y.eps)
        layer = _rows_layer(blocks[i], m, caches[i][0], types) \
            if i < len(blocks) else None
        if layer is None:
            # fp32 parts where a norm adds them up, as Transformer._blocks has it
            parts = i < len(blocks) and blocks[i].fuses_residual()
            return x, ext.decode_gemm_rows(h, down.ws, down.n, down.half,
                                           parts), i
        x, y = _add_rows(x, h, down, layer.blk.norm1)
