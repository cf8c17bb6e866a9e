"""Linear dispatch: which product runs on which kernel.

Products of up to 128 rows are bound by the weights; csrc/decode_gemm.hip streams
W at HBM rate where hipBLASLt's tiles measured 25-45% (profiles/). Above that
prompts and fine-tunes run on csrc/gemm_tiles.hip where there are too few tiles
for the library's, or where what follows the product can end it, and otherwise on
hipBLASLt via F.linear.
"""
from __future__ import annotations

import contextlib
import os
import threading
import weakref

import torch
import torch.nn.functional as F

from . import _backend

# The first tile kernel; superseded by decode_gemm (kept for A/B runs).
_USE_SKINNY = os.environ.get("RB_SKINNY_GEMM", "0") == "1"
# v2 weight-stream kernel (csrc/decode_gemm.hip): default-on; RB_DECODE_GEMM=0
# falls back to hipBLASLt.
_USE_DECODE_GEMM = os.environ.get("RB_DECODE_GEMM", "1") == "1"


# data_ptr(weight) -> (e4m3 bytes in the decode GEMM's order, f32 per-channel
# scale, distance of rows in pairs (below), the weight's version, weakref to the
# weight). Populated by quantize_fp8 (serving with MODEL_LOAD_IN_8BIT); looked up
# on the decode fast path.
_FP8_REGISTRY: dict[int, tuple] = {}

# data_ptr(weight) -> fragment-lane-major copy ([N/32][K/16][lane][8])
# consumed by csrc/decode_gemm.hip. A second full-precision weight copy:
# 288 GB HBM3E per GPU makes layout-specialized decode weights the right
# trade on MI355X (prefill/training keep the original [N,K] tensor).
# value: (swizzled copy, (N, K), distance of rows in pairs, the weight's version,
# weakref to the registered tensor). Pairs (csrc/decode_ends.h; 0: rows in order)
# let a product end in what follows it, a gated unit or a rotation.
# data_ptr alone is NOT a safe key — a freed weight's address gets
# recycled by later allocations, so every lookup verifies tensor
# identity through the weakref (stale entries are dropped lazily).
_DECODE_W_REGISTRY: dict[int, tuple] = {}


def _version(weight: torch.Tensor):
    return None if weight.is_inference() else weight._version


def _registry_get(reg: dict, weight: torch.Tensor):
    """A weight's entry, for all products alike: none once the weight has
    changed in place (changes through .data leave no trace). The entry stays,
    as a captured step may read its copy."""
    entry = reg.get(weight.data_ptr())
    if entry is None:
        return None
    if entry[-1]() is not weight:
        del reg[weight.data_ptr()]
        return None
    if entry[-2] != _version(weight):
        return None
    served = getattr(_RECORD, "weights", None)
    if served is not None:
        served[id(weight)] = weight
    return entry


_RECORD = threading.local()


@contextlib.contextmanager
def copies_read():
    """Within it, the weights of which this thread looked a copy up are
    gathered; afterwards the list holds a Versions of them."""
    _RECORD.weights, result = {}, []
    try:
        yield result
    finally:
        weights = list(_RECORD.weights.values())
        _RECORD.weights = None
    result.append(_backend.ext().Versions(
        [w for w in weights if not w.is_inference()]))


def register_decode_weight(weight: torch.Tensor, half: int = 0) -> None:
    """Build + register the decode-GEMM weight layout for `weight`; with `half`
    its rows go in pairs that far apart."""
    for ptr in [p for p, e in _DECODE_W_REGISTRY.items() if e[-1]() is None]:
        del _DECODE_W_REGISTRY[ptr]          # purge dead entries
    ws = _backend.ext().decode_swizzle_w(weight.data, half)
    _DECODE_W_REGISTRY[weight.data_ptr()] = (
        ws, (int(weight.shape[0]), int(weight.shape[1])), half,
        _version(weight), weakref.ref(weight))


E4M3_MAX = 448.0


def _fp8_served(n: int, k: int) -> bool:
    """Sizes of a weight that the fp8 decode GEMM takes."""
    return n % 64 == 0 and k % 256 == 0


@torch.no_grad()
def quantize_fp8(weight: torch.Tensor, half: int = 0
                 ) -> tuple[torch.Tensor, torch.Tensor]:
    """Row-wise (per-output-channel) OCP e4m3 quantization; registers the
    pair so fast_linear dispatches to the fp8 decode GEMM (`half`: as in
    register_decode_weight, of the copy that it reads). Pass the
    PERSISTENT tensor object (Parameter / fused buffer), not .data —
    lookups verify identity via weakref."""
    scale = weight.float().abs().amax(dim=1).clamp(min=1e-8) / E4M3_MAX
    w8 = (weight.float() / scale[:, None]).to(torch.float8_e4m3fn)
    w8_bytes = w8.view(torch.uint8).contiguous()
    served = (_backend.ext().decode_swizzle_w8(w8_bytes, half)
              if weight.is_cuda and _fp8_served(*weight.shape) else w8_bytes)
    _FP8_REGISTRY[weight.data_ptr()] = (served, scale.contiguous(), half,
                                        _version(weight), weakref.ref(weight))
    return w8_bytes, scale


def dequantize_fp8(w8_bytes: torch.Tensor, scale: torch.Tensor,
                   dtype=torch.bfloat16) -> torch.Tensor:
    return (w8_bytes.view(torch.float8_e4m3fn).float() *
            scale[:, None]).to(dtype)


def _swizzled(x: torch.Tensor, m: int, k: int) -> torch.Tensor:
    """x as the decode GEMM's operand: producers (rmsnorm_fwd_dec,
    *_packed_dec) attach it; otherwise one tiny kernel builds it here."""
    xs = getattr(x, "_rb_swz", None)
    return xs if xs is not None else _backend.ext().decode_swizzle_x(
        x.reshape(m, k).contiguous())


def fast_linear(x: torch.Tensor, weight: torch.Tensor,
                bias: torch.Tensor | None = None) -> torch.Tensor:
    if (bias is None and not torch.is_grad_enabled()
            and x.dtype == torch.bfloat16 and _backend.use_hip(x)
            and weight.is_contiguous()):
        k = x.shape[-1]
        m = x.numel() // k
        n = weight.shape[0]
        if m <= 32:
            if _fp8_served(n, k):
                q = _registry_get(_FP8_REGISTRY, weight)
                if q is not None:
                    y = _backend.ext().decode_gemm_fp8(
                        _swizzled(x, m, k), q[0], q[1], m, n, k, half=q[2])
                    return y.view(*x.shape[:-1], n)
            if _USE_DECODE_GEMM:
                dw = _registry_get(_DECODE_W_REGISTRY, weight)
                if dw is not None:
                    y = _backend.ext().decode_gemm(_swizzled(x, m, k), dw[0],
                                                   m, n, k, half=dw[2])
                    return y.view(*x.shape[:-1], n)
            if _USE_SKINNY and n % 64 == 0 and k % 256 == 0:
                y = _backend.ext().skinny_gemm(x.reshape(m, k).contiguous(),
                                               weight)
                return y.view(*x.shape[:-1], n)
        elif m <= 128:
            y = _rows_linear(x, weight, m, n, k)
            if y is not None:
                return y
        if (m > 32 and k > _LONG_ROW and n % 4 == 0 and x.dim() == 2 and
                -(-m // 256) * -(-n // 256) <= 144):
            # with few tiles the library is slow at such sums, as in
            # linear_f32_parts (us in one and in two, 3072 x 24576: 512 rows
            # 274 and 155, 1021 274 and 210, 3001 666 and 405; 5000 rows, 240
            # tiles, 541 in one)
            return _backend.ext().sum_parts(linear_f32_parts(x, weight))
    return F.linear(x, weight, bias)


def _rows_copy(x: torch.Tensor, weight: torch.Tensor, m: int, n: int, k: int):
    """The registered copy of `weight` where decode_gemm_rows takes x and it."""
    if not _USE_DECODE_GEMM or n % 32 or k % 16 or k < 1024 or \
            not x.is_contiguous() or x.data_ptr() % 16:
        return None
    return _registry_get(_DECODE_W_REGISTRY, weight)


def _rows_linear(x: torch.Tensor, weight: torch.Tensor, m: int, n: int,
                 k: int) -> torch.Tensor | None:
    """x @ weight^T of up to 128 rows on the decode GEMM that reads x as it is,
    or None where the weight has no decode layout.

    us on the library and there: 64 rows, 22016 x 4096 44.4 and 35.8, 4096 x
    4096 23.0 and 14.1, 4096 x 14336 40.4 and 27.3, 3072 x 24576 102 and 34; 128
    rows, 46.5 and 46.9, 26.9 and 17.6, 76.9 and 32.5, 133 and 43."""
    dw = _rows_copy(x, weight, m, n, k)
    if dw is None:
        return None
    y = _backend.ext().decode_gemm_rows(x.view(m, k), dw[0], n, dw[2])
    return y.view(*x.shape[:-1], n)


def _tiles_serve(x: torch.Tensor, weight: torch.Tensor, glu: bool = False
                 ) -> bool:
    """The tiles of csrc/gemm_tiles.hip take x, of more than 128 rows, for a
    result that is not differentiated."""
    return (x.is_cuda and x.dim() == 2 and x.shape[0] > 128 and
            x.dtype == torch.bfloat16 and not torch.is_grad_enabled() and
            _backend.ext().tile_gemm_takes(x, weight, glu))


def _rows_served(x: torch.Tensor, weight: torch.Tensor, least: int = 33):
    """_rows_copy for results that are not differentiated, of `least` to 128
    rows; up to 32 only where no 8-bit weights serve them."""
    if not (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and
            least <= x.shape[0] <= 128 and not torch.is_grad_enabled() and
            weight.is_contiguous()):
        return None
    if x.shape[0] <= 32 and _registry_get(_FP8_REGISTRY, weight) is not None:
        return None
    return _rows_copy(x, weight, x.shape[0], weight.shape[0], x.shape[1])


def rows_glu(x: torch.Tensor, weight: torch.Tensor, gelu: bool
             ) -> torch.Tensor | None:
    """act(x G^T) * (x U^T) of weight = [G ; U] and more than 32 rows in one
    launch, or None where nothing serves it: up to 128 rows a paired copy (us
    with the product and the gated unit apart and here, 64 rows: 22016 x 4096
    40.2 and 37.6, 49152 x 3072 64.5 and 59.1), above that tiles (22016 x 4096: 129
    rows 55 and 48, 512 91 and 77, 1537 247 and 233, 2048 298 and 270, 4500 623
    and 586; 28672 x 4096: 1400 277 and 283, 1800 354 and 337, 6500 1283 and
    1093; 49152 x 3072: 256 98 and 76, 1021 267 and 228, 3200 821 and 713; 11264 x 2048:
    900 55 and 40; 5632 x 1024: 129 15 and 12; 57344 x 8192: 256 243 and 244, 1536
    1083 and 1051, 4096 2613 and 2633. Of 200 sizes two were slower by more than 2%,
    1400 x 28672 x 4096 274 and 292 and 640 x 49152 x 3072 189 and 196)."""
    if _tiles_serve(x, weight, True):
        return _backend.ext().tile_gemm(x, weight, glu=2 if gelu else 1)
    dw, n = _rows_served(x, weight), weight.shape[0]
    if dw is None or dw[2] * 2 != n or \
            not _backend.ext().rows_ends_pay(x.shape[0], n, x.shape[1]):
        return None
    return _backend.ext().rows_glu(x, dw[0], n, gelu)


def rows_heads(x: torch.Tensor, weight: torch.Tensor, cos, sin, positions, kc,
               vc, slots, hq: int, rows: bool) -> torch.Tensor | None:
    """The product of 33 to 128 rows with joint weights of q, k and v whose
    rotation and cache write it does too: q [T, hq, dh], or, in rows, q, k and v
    side by side, also of fewer (a step of so few goes by decode_chain.py); None
    where no paired copy serves it."""
    dw, n = _rows_served(x, weight, 1 if rows else 33), weight.shape[0]
    if dw is None or kc.dtype != torch.bfloat16 or \
            dw[2] * 2 != kc.shape[3] or \
            not _backend.ext().rows_ends_pay(x.shape[0], n, x.shape[1]):
        return None
    return _backend.ext().rows_heads(x, dw[0], n, cos, sin, positions, kc, vc,
                                     slots, hq, rows)


def rows_parts(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor | None:
    """x @ weight^T of more than 32 rows for a norm that adds up parts of it
    (ops.rmsnorm_res): fp32 [P, T, N], or [T, N] where the kernel splits
    nothing; None where nothing serves it. us with the sum in a launch of its
    own and in the norm, 64 rows: 4096 x 4096 17.8 and 16.4, 4096 x 11008 29.3
    and 27.6.

    Above 128 rows in tiles, where these are few and so share the sums, or one
    round of them does (us with the norm, library and here: 4096 x 4096 129 rows
    31 and 19, 300 32 and 27, 512 34 and 31; 4096 x 14336 129 58 and 39, 512 97
    and 65, 1021 141 and 109, 2048 220 and 206; 3072 x 24576 512 151 and 90,
    1021 209 and 136, 2048 328 and 252; 8192 x 8192 512 87 and 74). Otherwise
    the library is as fast or faster (4096 x 4096 768 39 and 45, 8192 x 8192
    1280 147 and 157), as it is with short sums, where begin and end of a tile
    count for more (2048 x 2048 129 13 and 15, 400 16 and 19; 1024 x 2816 129 12
    and 15, 1021 19 and 21; but 3584 x 3584 300 29 and 23, 2048 x 5632 400 29 and 24).
    """
    if _tiles_serve(x, weight):
        (m, k), n = x.shape, weight.shape[0]
        if _sums_in_parts(m, n, k):
            return _backend.ext().tile_gemm(x, weight, max_parts=4)
        return _one_round(x, weight)
    dw = _rows_served(x, weight)
    return None if dw is None else _backend.ext().decode_gemm_rows(
        x, dw[0], weight.shape[0], dw[2], True)


def _sums_in_parts(m: int, n: int, k: int) -> bool:
    return k >= 3072 and _backend.ext().tile_gemm_parts(m, n, k) > 1


def _one_round(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor | None:
    """x @ weight^T of long rows in one round of tiles of 256 x 128, or None
    where the library is as good: it takes 192 or 256 columns, too few tiles for
    256 CUs (us there and here, to 4096 columns: 2048 rows of 11008 160 and 145,
    of 14336 205 and 193, of 20480 323 and 265, of 28672 367 and 394; to 3584 2048 of
    14336 190 and 175; to 5120 1536 of 13824 191 and 182; to 8192 1024 of 13824 194
    and 186, of 28672 446 and 397; to 14336 512 of 11008 167 and 156, 257 of 13824 152
    and 159. Outside: 2048 of 4096 58 and 58; 1280 of 11008 119 and 130)."""
    (m, k), n = x.shape, weight.shape[0]
    tiles = -(-m // 256) * -(-n // 128)
    if k > 8192 and 224 <= tiles <= 256 and m <= 2048 and \
            _backend.ext().tile_gemm_takes(x, weight):
        return _backend.ext().tile_gemm(x, weight)
    return None


def _whole_rounds(rows: int, cols: int) -> int:
    """Columns of a library product to be computed in a call of their own, a
    whole number of rounds of 256 x 256 tiles over the 256 CUs; the rest in a
    second one. `cols` where one call does for all.

    In one call the library leaves CUs idle in the last round, or takes a slower
    tile; the second call has a tile for what is left. us in one call and in
    two, inputs of 4096: 2048 rows x 22016 402 and 268, 4096 x 22016 636 and 506,
    2816 x 6144 216 and 111, 3001 x 28672 530 and 499, 8192 x 11008 643 and 503;
    3584 x 12288 256 and 257, 6000 x 4096 155 and 160. Up to 1280 rows it gives
    nothing on the whole (1024 x 22016 155 and 159, 1280 x 28672 239 and 230,
    1024 x 28672 183 and 189), nor where all tiles are whole rounds by
    themselves (6 x 128 tiles, 155 and 164)."""
    down, across = -(-rows // 256), -(-cols // 256)
    if down <= 5 or down > 256 or down * across % 256 == 0:
        return cols
    step = 256 // down
    return min(across // step * step * 256 or cols, cols)


def _differentiated(x: torch.Tensor, weight: torch.Tensor) -> bool:
    return torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad)


def wide_product(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """x @ weight^T on the GPU, in whole rounds of tiles; one call where the result
    is differentiated."""
    if _differentiated(x, weight):
        return x @ weight.t()
    rows, cols = x.shape[0], weight.shape[0]
    if _many_in_tiles(rows, cols, x.shape[1]) and \
            _backend.ext().tile_gemm_takes(x, weight):
        return _backend.ext().tile_gemm(x, weight)
    y = _one_round(x, weight)
    if y is not None:
        return y
    main = _whole_rounds(rows, cols)
    if main >= cols:
        return x @ weight.t()
    y = x.new_empty(rows, cols)
    torch.mm(x, weight[:main].t(), out=y[:, :main])
    torch.mm(x, weight[main:].t(), out=y[:, main:])
    return y


def _wide_in_tiles(m: int, n: int, k: int) -> bool:
    """Whether wide weights' product of few rows runs in own tiles: one row of
    tiles of 256, or a second one that is nearly as good (us in the library and
    in tiles: 12288 x 4096 129 rows 38 and 36, 256 48 and 43, 320 51 and 47;
    12288 x 3072 192 33 and 32, 320 42 and 40; 15360 x 5120 256 64 and 59, 320 60
    and 64; 18432 x 3072 256 51 and 45; 12288 x 1024 256 17 and 16, 320 17 and 18).
    Wider ones the library takes in whole rounds (24576 x 4096 192 58 and 60,
    320 72 and 79; 32768 x 1024 320 26 and 31; 24576 x 8192 129 100 and 119), of
    narrower ones there are too few tiles (6144 x 4096 200 25 and 34)."""
    return 12288 <= n < 20480 and \
        (m <= 256 or (m <= 320 and n < 15360 and 2048 <= k < 8192))


def _many_in_tiles(m: int, n: int, k: int) -> bool:
    """The same of more rows (tile_gemm_pays in csrc/gemm_tiles.hip)."""
    return m > 320 and _backend.ext().tile_gemm_pays(m, n, k)


def wide_linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """fast_linear of rows x that are there also where they have a decode operand;
    of many rows a wide_product. A result that is differentiated is fast_linear's.

    From 17 to 32 rows the kernel that shares x is the faster one where it has
    about one workgroup for every CU (us without and with it, 32 rows: 22016 x
    4096 34.9 and 31.2, 12288 x 4096 23.2 and 21.7; 49152 x 3072 52.7 and 53.0,
    6144 x 4096 15.9 and 15.4, of 24 rows 47.9 and 52.6, 14.7 and 15.0)."""
    if x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and \
            not _differentiated(x, weight):
        (m, k), n = x.shape, weight.shape[0]
        if (_wide_in_tiles(m, n, k) or _many_in_tiles(m, n, k)) and \
                _tiles_serve(x, weight):
            return _backend.ext().tile_gemm(x, weight)
        if m > 1280:
            return wide_product(x, weight)
        if 16 < m <= 32 and 10240 <= n <= 32768 and \
                _registry_get(_FP8_REGISTRY, weight) is None:
            y = _rows_linear(x, weight, m, n, k)
            if y is not None:
                return y
    return fast_linear(x, weight)


def _lora_in_tiles(m: int, n: int, k: int) -> bool:
    """Whether a product that adapters' parts are added to runs in tiles that end
    with them, or in the library with a pass over its result.

    Rows of up to 5120: where the result is wide or has more than 32 tiles of 256 x
    256 (us in the library with the pass and in tiles: 12288 x 4096 129 rows 44 and
    38, 2048 169 and 169, 3001 251 and 232; 6144 x 4096 129 44 and 34, 3001 143 and
    135; 22016 x 4096 700 149 and 127, 2300 359 and 334; 28672 x 4096 2048 385 and
    364; 27648 x 5120 1536 393 and 346; 4096 x 4096 900 42 and 36, 512 34 and 39;
    2048 x 2048 1800 25 and 20), of up to 60 million results (_large_lora_in_tiles).

    Longer rows: where one round of tiles does (4096 x 11008 1800 158 and 139, 2048
    164 and 146, 3001 209 and 201; 4096 x 14336 2048 205 and 185; 5120 x 13824 1536
    190 and 175; 8192 x 8192 1024 123 and 111). With fewer tiles CUs are idle for
    long (4096 x 14336 512 94 and 136, 1280 152 and 166, 2048 x 5632 1024 42 and 57),
    with more the library is as fast (4096 x 14336 4096 320 and 333, 8192 x 28672
    700 288 and 348)."""
    def tiles(rows, cols):
        return -(-m // rows) * -(-n // cols)
    if m <= 128 or n < 2048 or m * n > 60_000_000:
        return False
    if k <= 5120:
        return n >= 6144 or tiles(256, 256) > 32
    return k <= 16384 and n >= 4096 and \
        any(224 <= t <= 256 for t in (tiles(256, 128), tiles(192, 256)))


def _large_lora_in_tiles(m: int, n: int, k: int) -> bool:
    """The same of results of more than 60 million (us in the library with the pass and
    in tiles: 22016 x 4096 3001 rows 447 and 430, 8192 1129 and 1072; 28672 x 4096 2300
    420 and 387, 3001 564 and 543, 8192 1438 and 1342; 27648 x 5120 4096 915 and 825;
    12288 x 4096 8192 631 and 608; 11264 x 2048 6000 257 and 241; a step of mistral-7b,
    3001 tokens, 97.7 ms and 96.1). Of 347 sizes, to 24000 rows and 57344 columns, one
    is slower by 3%, the mean is 0.81."""
    return m * n > 60_000_000 and n >= 6144 and 256 <= k <= 5120


def wide_product_lora(x: torch.Tensor, weight: torch.Tensor, t: torch.Tensor,
                      bs: list, scale: float) -> torch.Tensor:
    """wide_product(x, weight) + scale t_i B_i^T of adapters side by side
    (csrc/lora_group.hip)."""
    ext, (n, k) = _backend.ext(), weight.shape
    m = x.shape[0]
    if (_lora_in_tiles(m, n, k) or _large_lora_in_tiles(m, n, k)) and \
            ext.tile_gemm_takes(x, weight):
        return ext.tile_lora(x, weight, t, bs, scale)
    y = wide_product(x, weight)
    ext.lora_add_(y, t, bs, scale, False)
    return y


def wide_product_grad(dy: torch.Tensor, weight: torch.Tensor,
                      dt: torch.Tensor | None = None, As=()) -> torch.Tensor:
    """dy @ weight on the GPU, weight [N, K], and + dt_i A_i of adapters side by
    side: in tiles (csrc/gemm_tiles.hip), which take the adapters along, where they
    are as good as the library and a pass over its result."""
    ext, (n, k) = _backend.ext(), weight.shape
    if dy.is_contiguous() and ext.tile_gemm_down_pays(dy.shape[0], k, n) and \
            ext.tile_gemm_down_takes(dy, weight):
        t = dt if dt is not None else dy.new_empty(0, dy.shape[0], 16)
        dx = ext.tile_gemm_down(dy, weight, t, list(As), max_parts=4)
        return dx if dx.dim() == 2 else ext.sum_parts(dx)
    dx = _library_grad(dy, weight)
    if dt is not None:
        ext.lora_add_(dx, dt, list(As), 1.0, True)
    return dx


def _library_grad(dy: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """Wide results in whole rounds of tiles, like wide_product's (2048 rows of
    4096 to 11008 columns: 284 and 171 us; to 4096 and 6144 columns 3 to 14%
    slower in two calls). Long sums with few tiles in two fp32 halves, rounded
    once: there the library keeps tiles of 256 x 256, of which there are not
    enough (us in one sum and in two, to 4096 columns: 2048 rows of 22016 453
    and 372, 512 213 and 163, 1024 rows of 28672 359 and 307, 2048 401 and 463;
    2049 rows of 17408 325 and 300, 2304 367 and 314; with more tiles, 2560 rows
    of 22016, 372 and 390; of 12288 and 2048 rows 195 and 213). From 60 to 2300
    rows two are 20% faster of 22016, 17% of 24576 to 3072 columns, 5% of 28672,
    and 11% slower of 49152 to 3072 (1024 rows 435 and 516, 2048 523 and 885)."""
    rows, (n, k) = dy.shape[0], weight.shape
    if k >= 8192:
        main = _whole_rounds(rows, k)
        if main < k:
            dx = dy.new_empty(rows, k)
            torch.mm(dy, weight[:, :main], out=dx[:, :main])
            torch.mm(dy, weight[:, main:], out=dx[:, main:])
            return dx
    if 16384 < n <= 32768 and k % 4 == 0 and \
            -(-rows // 256) * -(-k // 256) <= 144:
        half = n // 128 * 64
        parts = torch.empty(2, rows, k, dtype=torch.float32, device=dy.device)
        for part, at in zip(parts, (slice(0, half), slice(half, n))):
            torch.mm(dy[:, at], weight[at], out_dtype=torch.float32, out=part)
        return _backend.ext().sum_parts(parts)
    return dy @ weight


def decode_linear_raw(x, weight, f32: bool = False):
    """Decode GEMM that may return an UNCOMBINED fp32 split-K slab
    [split, M, N] (consumer kernels fold it — rmsnorm_res_slab_fwd_dec),
    or a plain bf16 [M, N]; with f32=True always the slab (of one slice
    where the product is not split). Falls back to fast_linear when the
    weight has no registered decode layout. Returns (out, is_slab)."""
    k = x.shape[-1]
    m = x.numel() // k
    n = weight.shape[0]
    q = None if f32 or not _fp8_served(n, k) else \
        _registry_get(_FP8_REGISTRY, weight)
    if q is not None and m <= 32 and x.dtype == torch.bfloat16:
        out = _backend.ext().decode_gemm_fp8(_swizzled(x, m, k), q[0], q[1],
                                             m, n, k, True, q[2])
        return out, out.dtype == torch.float32
    dw = _registry_get(_DECODE_W_REGISTRY, weight)
    if dw is None or not _USE_DECODE_GEMM:
        with torch.no_grad():
            return fast_linear(x, weight), False
    xs = _swizzled(x, m, k)
    out = _backend.ext().decode_gemm_raw(xs, dw[0], m, n, k, f32, dw[2])
    return out, out.dtype == torch.float32


class Copy:
    """What the decode products of up to 32 rows read of a weight [n, k]."""

    def __init__(self, weight: torch.Tensor):
        self.n, self.k = weight.shape
        q = _registry_get(_FP8_REGISTRY, weight) \
            if _fp8_served(self.n, self.k) else None
        dw = _registry_get(_DECODE_W_REGISTRY, weight) \
            if q is None and _USE_DECODE_GEMM else None
        self.fp8 = q is not None
        self.ws, self.scale, self.half = \
            (q[0], q[1], q[2]) if self.fp8 else \
            (dw[0], None, dw[2]) if dw is not None else (None, None, 0)

    def shares_x(self, m: int) -> bool:
        """From 17 rows the kernel that shares x between workgroups' waves wins
        where it has about one workgroup for every CU (wide_linear)."""
        return 16 < m <= 32 and not self.fp8 and 10240 <= self.n <= 32768

    def product(self, xs, m: int):
        """Of an operand: bf16 [m, n], or fp32 parts [P, m, n] of it."""
        ext = _backend.ext()
        if self.fp8:
            return ext.decode_gemm_fp8(xs, self.ws, self.scale, m, self.n,
                                       self.k, True, self.half)
        return ext.decode_gemm_raw(xs, self.ws, m, self.n, self.k,
                                   half=self.half)


def few_rows_mlp(x: torch.Tensor, weight: torch.Tensor, down: torch.Tensor,
                 gelu: bool, raw: bool) -> torch.Tensor | None:
    """act(x G^T) * (x U^T) D^T of weight = [G ; U] and up to 32 rows, the gated
    unit as the end of the first product; with `raw` possibly fp32 parts of it;
    None where there are no copies for it.

    A product of a paired copy that ends in nothing is slower than one of a copy in
    order, for its columns go to memory in pieces of 32 bytes (us of 16 and 32
    rows: 49152 x 3072 48.3 and 58.4, 46.3 and 53.1 in order; 22016 x 4096 32.0 and
    36.3, 32.8 and 35.4)."""
    if not (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and
            1 <= x.shape[0] <= 32 and not torch.is_grad_enabled() and
            weight.is_contiguous() and down.is_contiguous()):
        return None
    first, second = Copy(weight), Copy(down)
    if first.ws is None or second.ws is None or first.half * 2 != first.n:
        return None
    ext, (m, k) = _backend.ext(), x.shape
    if first.shares_x(m) and x.is_contiguous() and x.data_ptr() % 16 == 0:
        h = ext.rows_glu(x, first.ws, first.n, gelu, True)
    else:
        h = ext.decode_glu(_swizzled(x, m, k), first.ws, first.scale, m,
                           first.n, k, gelu)
    y = second.product(h, m)
    return y if raw or y.dtype != torch.float32 else ext.sum_parts(y)


def decode_ready(weight: torch.Tensor, m: int) -> bool:
    """True when a product of m rows with `weight` runs on the decode GEMM
    (so that its producer should emit the swizzled operand)."""
    return (m <= 32 and _USE_DECODE_GEMM and weight.is_cuda and
            _registry_get(_FP8_REGISTRY, weight) is None and
            _registry_get(_DECODE_W_REGISTRY, weight) is not None)


def decode_operand(m: int, k: int, like: torch.Tensor) -> torch.Tensor:
    """Buffer for a decode-GEMM operand of m <= 32 rows and k columns,
    [k/16][2][32][8] (filled by the kernels that produce the rows)."""
    return torch.empty((k // 16) * 512, dtype=like.dtype, device=like.device)


def linear_f32(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """x @ weight^T with the fp32 accumulator as the result."""
    if x.is_cuda and x.dtype == torch.bfloat16:
        return torch.mm(x, weight.t(), out_dtype=torch.float32)
    return F.linear(x, weight).float()


# Row length beyond which hipBLASLt's choice is often poor: 300 to 570 us by
# the number of rows around 2048, where two products of half the length
# together take about 310 us at each.
_LONG_ROW = 16384


def linear_f32_parts(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """linear_f32 for a consumer that takes several parts: [T, N], or, of
    long rows, [2, T, N] to be summed."""
    K = x.shape[1]
    if not (x.is_cuda and x.dtype == torch.bfloat16 and K > _LONG_ROW):
        return linear_f32(x, weight)
    out = torch.empty(2, x.shape[0], weight.shape[0], dtype=torch.float32,
                      device=x.device)
    half = K // 128 * 64
    for o, at in zip(out, (slice(0, half), slice(half, K))):
        torch.mm(x[:, at], weight[:, at].t(), out_dtype=torch.float32, out=o)
    return out


class Linear(torch.nn.Linear):
    """nn.Linear with the decode-GEMM fast path."""

    def forward(self, x):
        return fast_linear(x, self.weight, self.bias)
