"""LoRA adapters (Hu et al. 2021) over the transformer's linear layers.

The reference platform's fine-tune path is LoRA via the external HF
trainer image (reference examples/llama2-7b/finetuned-model.yaml); here it
is native: frozen base weights, trainable low-rank A/B pairs on the
attention + MLP projections. Three ways, by what a layer is:

* rank 16, bf16, no bias, on the GPU (_LoRAPacked): siblings that share
  their input side by side, one product with the frozen weights each way
  (csrc/gemm_tiles.hip), the adapters' other products on kernels of
  csrc/lora_group.hip that read x, y and dy once for all of them;
* other layers without bias (_LoRAFused, _LoRAFusedT): library products,
  both gradient merges in place (the eager formulation measured ~450 extra
  elementwise launches per llama2-7b step);
* the rest (bias, dropout, sharded): the composite, by autograd.
"""
from __future__ import annotations

import math
import os

import torch
from torch import nn

from ..ops import _backend
from ..ops.linear import wide_product_grad, wide_product_lora
from ..parallel.tp import ColumnParallelLinear, RowParallelLinear
from ..utils.modules import plain


def _delta_add_(y, t, w, scale, w_transposed=True):
    """y += scale * t @ (w^T if w_transposed else w).

    r=16 w_transposed merges run the MFMA lora_badd_ kernel (both
    operands are natural contiguous 32x32x16 fragments; hipBLASLt runs
    these K=16 accumulates ~4x off the y-stream roofline — r33
    torch.profiler). RB_LORA_MFMA=0 reverts to in-place addmm_.
    The older scalar lora_delta_ kernel (per-lane W gather, measured
    slower) stays behind RB_LORA_KERNEL=1 for A/B work only."""
    if (os.environ.get("RB_LORA_MFMA", "1") == "1"
            and y.is_cuda and y.dtype == torch.bfloat16
            and t.shape[1] == 16 and y.shape[1] % 32 == 0
            and w.dtype == torch.bfloat16):
        from ..ops import _backend
        if _backend.use_hip(y):
            # w_transposed=False (y += t @ w, w [16, N]): transpose the
            # TINY w into the kernel's [N, 16] fragment layout — ~5 us
            # vs the 110 us hipBLASLt accumulate it replaces (r35
            # profile, [2048, 11008] dx merge).
            wk = w if w_transposed else w.t()
            _backend.ext().lora_badd_(y, t.contiguous(), wk.contiguous(),
                                      scale)
            return y
    if (os.environ.get("RB_LORA_KERNEL", "0") == "1"
            and y.is_cuda and y.dtype == torch.bfloat16
            and y.shape[1] % 8 == 0
            and t.shape[1] <= 32 and t.shape[1] % 8 == 0):
        from ..ops import _backend
        _backend.ext().lora_delta_(y, t.contiguous(), w.contiguous(),
                                   scale, w_transposed)
        return y
    return y.addmm_(t, w.t() if w_transposed else w, alpha=scale)

DEFAULT_TARGETS = ("q_proj", "k_proj", "v_proj", "o_proj",
                   "gate_proj", "up_proj", "down_proj", "fc1", "fc2")


# RB_EXPERIMENTAL_GEMM=1 routes the big frozen-weight GEMMs through the
# 8-phase 256^2 kernel (ops/csrc/gemm_train.hip) instead of hipBLASLt.
# The dgrad (dy @ W) is NN-shaped, so frozen weights get a one-time
# transposed copy (cheap next to 288 GB HBM) and run as NT(dy, W^T).
_USE_CUSTOM_GEMM = os.environ.get("RB_EXPERIMENTAL_GEMM", "0") == "1"
_WT_CACHE: dict[int, torch.Tensor] = {}


def _nt_ok(m: int, n: int, k: int) -> bool:
    return m % 256 == 0 and n % 256 == 0 and k % 128 == 0


def _nt(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a[M,K] @ b[N,K]^T — custom kernel when eligible, else hipBLASLt."""
    if (_USE_CUSTOM_GEMM and a.is_cuda and a.dtype == torch.bfloat16
            and _nt_ok(a.shape[0], b.shape[0], a.shape[1])):
        from ..ops import _backend
        return _backend.ext().train_gemm_nt(a.contiguous(), b.contiguous())
    return a @ b.t()


def _wt(w: torch.Tensor) -> torch.Tensor:
    wt = _WT_CACHE.get(w.data_ptr())
    if wt is None:
        wt = w.t().contiguous()
        _WT_CACHE[w.data_ptr()] = wt
    return wt


class _LoRAGroupPrep(torch.autograd.Function):
    """tcat = x @ cat(A_1..A_n)^T for sibling adapters sharing the same
    input (q/k/v; gate/up): one activation stream instead of n.

    Backward: dcat = dtcat^T x (one GEMM, x read once) sliced into the
    per-adapter dA's, and dx = dtcat @ catA (one GEMM; autograd adds it
    to the base-path dx's)."""

    @staticmethod
    def forward(ctx, x, *As):
        catA = torch.cat(As)                    # [n*r, in]
        t = x @ catA.t()                        # [T, n*r]
        ctx.save_for_backward(x, catA)
        ctx.rs = [a.shape[0] for a in As]
        return t

    @staticmethod
    def backward(ctx, dt):
        x, catA = ctx.saved_tensors
        dcat = dt.t() @ x                       # [n*r, in]
        dx = dt @ catA
        das, off = [], 0
        for r in ctx.rs:
            das.append(dcat[off:off + r])
            off += r
        return (dx, *das)


class _LoRAGroup:
    """Shared-input sibling adapters + the per-forward tcat cache (of the
    input that it holds; dropped after every member consumed it so no
    autograd graph outlives the step)."""

    def __init__(self, members):
        self.members = members
        self._x = None
        self._t = None
        self._left = 0

    def packed(self, x):
        """All members' results on x side by side, or None where the members
        have to be called one by one."""
        if plain(LoRALinear, *self.members) and _packs(self.members, x):
            return _packed(self.members, x)
        return None

    def t_for(self, member, x):
        if self._x is not x or self._left <= 0:
            self._t = _LoRAGroupPrep.apply(
                x, *[m.lora_a for m in self.members])
            self._x = x
            self._left = len(self.members)
        i = self.members.index(member)
        off = sum(m.r for m in self.members[:i])
        t = self._t[:, off:off + member.r]
        self._left -= 1
        if self._left == 0:
            self._t = None
            self._x = None
        return t


class _LoRAFusedT(torch.autograd.Function):
    """y = x W^T + s t B^T with t precomputed by the group prep.
    dt flows back through _LoRAGroupPrep (which owns the dx merge and
    the dA GEMM for the whole group)."""

    @staticmethod
    def forward(ctx, x, w, t, b, scale):
        y = _nt(x, w)
        _delta_add_(y, t, b, scale)
        ctx.save_for_backward(w, t, b, x)
        ctx.scale = scale
        return y

    @staticmethod
    def backward(ctx, dy):
        w, t, b, x = ctx.saved_tensors
        s = ctx.scale
        if (_USE_CUSTOM_GEMM and dy.is_cuda and dy.dtype == torch.bfloat16
                and _nt_ok(dy.shape[0], w.shape[1], dy.shape[1])):
            dx = _nt(dy, _wt(w))
        else:
            dx = dy @ w
        dt = (dy @ b).mul_(s)
        db = torch.mm(dy.t(), t).mul_(s)
        return dx, None, dt, db, None


class _LoRAFused(torch.autograd.Function):
    """y = x W^T + s (x A^T) B^T with a GEMM-only backward.

    Eager autograd over the same math spends ~450 extra elementwise
    kernels per llama2-7b step on grad merges (profiles/). Here both
    merge points are addmm epilogues:
      dx = dy W  (+)= s (dy B) A     one addmm
      dA = s t2^T x,  dB = s dy^T t,  with t = x A^T, t2 = dy B
    The frozen base weight gets no wgrad at all.
    """

    @staticmethod
    def forward(ctx, x, w, a, b, scale):
        t = x @ a.t()                       # [T, r]
        # in-place addmm_: the out-of-place form first COPIES its beta
        # input (measured 448 DtoD copies x 8.2 us per train step, r11
        # torch.profiler); y is fresh from the base GEMM so accumulating
        # into it is safe
        y = _nt(x, w)
        _delta_add_(y, t, b, scale)
        ctx.save_for_backward(x, w, a, b, t)
        ctx.scale = scale
        return y

    @staticmethod
    def backward(ctx, dy):
        x, w, a, b, t = ctx.saved_tensors
        s = ctx.scale
        t2 = dy @ b                         # [T, r]
        if (_USE_CUSTOM_GEMM and dy.is_cuda and dy.dtype == torch.bfloat16
                and _nt_ok(dy.shape[0], w.shape[1], dy.shape[1])):
            dx = _nt(dy, _wt(w))
        else:
            dx = dy @ w
        _delta_add_(dx, t2, a, s, w_transposed=False)
        da = torch.mm(t2.t(), x).mul_(s)
        db = torch.mm(dy.t(), t).mul_(s)
        return dx, None, da, db, None


class _LoRAPacked(torch.autograd.Function):
    """y = x W^T + s (x A_i^T) B_i^T for siblings side by side (W and y by
    columns), or for one adapter: one product with the frozen weights each way,
    which the adapters' end, and their other products on kernels that read x and dy
    once for all of them (csrc/lora_group.hip)."""

    @staticmethod
    def forward(ctx, x, w, scale, n, *ab):
        ext = _backend.ext()
        t = ext.lora_down(x, list(ab[:n]))
        y = wide_product_lora(x, w, t, list(ab[n:]), scale)
        ctx.save_for_backward(x, w, t, *ab)
        ctx.scale, ctx.n = scale, n
        return y

    @staticmethod
    def backward(ctx, dy):
        ext, n = _backend.ext(), ctx.n
        x, w, t, *ab = ctx.saved_tensors
        As, Bs = list(ab[:n]), list(ab[n:])
        dy = dy.contiguous()
        if dy.data_ptr() % 16:      # a caller's own gradient may start anywhere
            dy = dy.clone()
        widths = [b.shape[0] for b in Bs]
        dt = ext.lora_down_columns(dy, Bs, ctx.scale)
        db, da = ext.lora_grads(dy, t, x, dt, widths, ctx.scale)
        db, da = db.split(widths), da.chunk(n)
        dx = None
        if ctx.needs_input_grad[0]:
            dx = wide_product_grad(dy, w, dt, As)
        return (dx, None, None, None, *da, *db)


def _packs(members, x) -> bool:
    """True when _LoRAPacked's kernels take these adapters on x, of which the
    weights have to be side by side in memory (_lay_side_by_side). What never
    changes comes first: a layer that is refused for its bias or its rank pays
    for little else."""
    for m in members:
        if m.r != 16 or getattr(m.base, "bias", None) is not None:
            return False
    if not x.is_cuda or x.dtype != torch.bfloat16 or x.dim() != 2 or \
            not x.is_contiguous() or x.data_ptr() % 16 or \
            not 0 < x.shape[0] <= 1 << 22 or _USE_CUSTOM_GEMM or \
            len(members) > 3 or os.environ.get("RB_LORA_MFMA", "1") != "1":
        return False
    for m in members:
        w = m.base.weight
        if (m.scale != members[0].scale or
                (m.dropout is not None and m.training) or
                not (isinstance(m.base, nn.Linear) or
                     getattr(m.base, "tp", 1) == 1) or
                w.requires_grad or w.dtype != torch.bfloat16 or
                not w.is_contiguous() or w.shape[0] % 64 or w.shape[1] % 64 or
                w.shape[1] != x.shape[1]):
            return False
        for p in (m.lora_a, m.lora_b):
            if p.dtype != torch.bfloat16 or not p.is_contiguous() or \
                    p.data_ptr() % 16:
                return False
    return _side_by_side(members) and _backend.use_hip(x)


def _side_by_side(members) -> bool:
    ws = [m.base.weight for m in members]
    return all(a.untyped_storage().data_ptr() == b.untyped_storage().data_ptr()
               and a.data_ptr() + a.numel() * a.element_size() == b.data_ptr()
               for a, b in zip(ws, ws[1:]))


@torch.no_grad()
def _lay_side_by_side(members) -> None:
    """Makes the members' frozen weights slices of one matrix."""
    ws = [m.base.weight for m in members]
    if not all(w.is_cuda and w.dim() == 2 and w.shape[1] == ws[0].shape[1] and
               w.dtype == ws[0].dtype and w.device == ws[0].device and
               w.untyped_storage().nbytes() == w.numel() * w.element_size()
               for w in ws):
        return
    whole = torch.cat([w.detach() for w in ws])
    for w, part in zip(ws, whole.split([w.shape[0] for w in ws])):
        w.data = part


def _packed(members, x):
    ws = [m.base.weight for m in members]
    rows, cols = sum(w.shape[0] for w in ws), ws[0].shape[1]
    w = ws[0].detach().as_strided((rows, cols), (cols, 1))
    return _LoRAPacked.apply(x, w, members[0].scale,
                             len(members), *(m.lora_a for m in members),
                             *(m.lora_b for m in members))


class LoRALinear(nn.Module):
    """Wraps a (possibly TP-sharded) linear: y = base(x) + scale * B(A(x)).

    A: [r, in_shard], B: [out_shard, r] — sharded the same way as the base
    weight so TP stays consistent; A/B are the only trainable params.
    """

    def __init__(self, base: nn.Module, r: int = 16, alpha: int = 32,
                 dropout: float = 0.0, dtype=None):
        super().__init__()
        self.base = base
        self.dropout = nn.Dropout(dropout) if dropout > 0 else None
        w = base.weight
        out_f, in_f = w.shape
        dtype = dtype or w.dtype
        self.r = r
        self.scale = alpha / r
        self.lora_a = nn.Parameter(torch.empty(r, in_f, dtype=dtype, device=w.device))
        self.lora_b = nn.Parameter(torch.zeros(out_f, r, dtype=dtype, device=w.device))
        nn.init.kaiming_uniform_(self.lora_a, a=math.sqrt(5))
        base.weight.requires_grad_(False)
        if getattr(base, "bias", None) is not None and isinstance(base.bias, nn.Parameter):
            base.bias.requires_grad_(False)

    def forward(self, x):
        base = self.base
        group = getattr(self, "_group", None)
        # siblings run one way: t_for counts on a call of each
        if all(_packs([m], x) for m in (group.members if group else (self,))):
            return _packed([self], x)
        if self.dropout is not None and self.training:
            # dropout on the adapter input (PEFT semantics) breaks the
            # single-addmm fusion; let autograd handle the composite
            y = self.base(x)
            t = torch.nn.functional.linear(self.dropout(x), self.lora_a)
            out_f = y.shape[-1]
            return torch.addmm(y.reshape(-1, out_f),
                               t.reshape(-1, self.r), self.lora_b.t(),
                               beta=1.0, alpha=self.scale).view(y.shape)
        if (isinstance(base, nn.Linear) or
                (getattr(base, "tp", 1) == 1 and base.bias is None)) and \
                x.dim() == 2 and getattr(base, "bias", None) is None:
            if group is not None:
                # shared-input siblings (q/k/v, gate/up): the A-GEMM,
                # its dA and the t-path dx merge run ONCE per group
                t = group.t_for(self, x)
                return _LoRAFusedT.apply(x, base.weight, t, self.lora_b,
                                         self.scale)
            # fully-fused fwd+bwd path: every product is one hipBLASLt
            # call, the two gradient merges ride addmm epilogues
            return _LoRAFused.apply(x, base.weight, self.lora_a,
                                    self.lora_b, self.scale)
        y = self.base(x)
        # adapter fused into the second GEMM's epilogue:
        # y = 1*y + scale * (x A^T) B^T — addmm keeps it in hipBLASLt,
        # no materialized adapter tensor, no separate mul/add kernels.
        t = torch.nn.functional.linear(x, self.lora_a)
        out_f = y.shape[-1]
        return torch.addmm(y.reshape(-1, out_f), t.reshape(-1, self.r),
                           self.lora_b.t(), beta=1.0,
                           alpha=self.scale).view(y.shape)

    @property
    def weight(self):  # so init / inspection code keeps working
        return self.base.weight


def apply_lora(model: nn.Module, r: int = 16, alpha: int = 32,
               dropout: float = 0.0, targets=DEFAULT_TARGETS) -> list[str]:
    """Freeze the model and wrap target linears with LoRA. Returns wrapped
    module names."""
    for p in model.parameters():
        p.requires_grad_(False)
    wrapped = []
    group_on = os.environ.get("RB_LORA_GROUP", "1") != "0"
    for name, module in model.named_modules():
        for child_name, child in list(module.named_children()):
            if child_name in targets and isinstance(
                    child, (nn.Linear, ColumnParallelLinear, RowParallelLinear)):
                setattr(module, child_name,
                        LoRALinear(child, r=r, alpha=alpha, dropout=dropout))
                wrapped.append(f"{name}.{child_name}" if name else child_name)
        if group_on and dropout <= 0:
            # group shared-input siblings for the one-A-GEMM path; only
            # plain bias-free nn.Linear bases (the fused-path criteria)
            for names in (("q_proj", "k_proj", "v_proj"),
                          ("gate_proj", "up_proj")):
                ms = [getattr(module, n, None) for n in names]
                if all(isinstance(m, LoRALinear) and
                       (isinstance(m.base, nn.Linear)
                        or getattr(m.base, "tp", 1) == 1) and
                       getattr(m.base, "bias", None) is None for m in ms):
                    _lay_side_by_side(ms)
                    g = _LoRAGroup(ms)
                    for m in ms:
                        m._group = g
    if not wrapped:
        raise ValueError("apply_lora: no target modules found")
    return wrapped


def lora_state_dict(model: nn.Module) -> dict[str, torch.Tensor]:
    return {k: v for k, v in model.state_dict().items()
            if "lora_a" in k or "lora_b" in k}


def merge_lora(model: nn.Module) -> None:
    """Fold adapters into base weights (for serving a fine-tuned model)."""
    for module in model.modules():
        if isinstance(module, LoRALinear):
            with torch.no_grad():
                delta = (module.lora_b.float() @ module.lora_a.float())
                module.base.weight.add_(delta.to(module.base.weight.dtype),
                                        alpha=module.scale)
                module.lora_b.zero_()
