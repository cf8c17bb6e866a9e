"""Decode products with what follows them in the same kernel (csrc/decode_ends.h,
csrc/decode_res.hip), and the steps of a model that run on them."""
import dataclasses

import pytest
import torch

from runbooks_amd import ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# one rounding to bf16 (half a unit of 8 bits), fp32 sums and exponentials
BF16 = 2 ** -8 + 1e-4


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _rows(operand, cols, m):
    return operand.view(cols // 16, 2, 32, 8).permute(2, 0, 1, 3) \
        .reshape(32, cols)[:m]


def _weight(n, k, half, fp8):
    """The copy that kernels read, its scales, and its values."""
    w = torch.randn(n, k, device=DEV).bfloat16()
    if not fp8:
        return ops.ext().decode_swizzle_w(w, half), None, w.double()
    w8 = w.to(torch.float8_e4m3fn)
    scale = torch.rand(n, device=DEV) + 0.5
    return (ops.ext().decode_swizzle_w8(w8.view(torch.uint8), half), scale,
            w8.double() * scale.double()[:, None])


def _squares(x, parts):
    """Sums of squares of x's rows in `parts` uneven parts."""
    share = torch.rand(x.shape[0], parts, device=DEV)
    share /= share.sum(1, keepdim=True)
    return share * x.float().square().sum(1, keepdim=True)


def _inverse_rms(x):
    return (x.double().square().mean(1, keepdim=True) + 1e-5).rsqrt()


def _act(g, gelu):
    return torch.nn.functional.gelu(g, approximate="tanh") if gelu else \
        torch.nn.functional.silu(g)


@pytest.mark.parametrize("m", [1, 5, 16, 17, 32])
@pytest.mark.parametrize("inter,k,parts", [(16, 1024, None), (48, 1056, 4),
                                           (5504, 4096, 256)])
@pytest.mark.parametrize("fp8,gelu", [(False, False), (False, True),
                                      (True, False)])
def test_gated_unit(m, inter, k, parts, fp8, gelu):
    torch.manual_seed(m + inter)
    ws, scale, w = _weight(2 * inter, k, inter, fp8)
    x = (torch.randn(m, k, device=DEV) / k ** 0.5).bfloat16()
    squares = None if parts is None else _squares(x, parts)
    f = 1.0 if parts is None else _inverse_rms(x)
    y = f * (x.double() @ w.t())
    ref = _act(y[:, :inter], gelu) * y[:, inter:]
    e = ops.ext()
    h = e.decode_glu(e.decode_swizzle_x(x), ws, scale, m, 2 * inter, k, gelu,
                     squares, 1e-5)
    assert _rel(_rows(h, inter, m), ref) < BF16
    if not fp8:
        h = e.rows_glu(x, ws, 2 * inter, gelu, True, squares, 1e-5)
        assert _rel(_rows(h, inter, m), ref) < BF16


@pytest.mark.parametrize("m", [1, 15, 16, 17])
@pytest.mark.parametrize("n,k,fp8", [
    (64, 1040, False), (64, 1056, False), (4096, 1088, False),
    (64, 1056, True), (64, 1088, True), (4096, 4160, True), (96, 64, True),
    # two to six chunks of a wave, whole and not, and e4m3 sums of one
    (64, 1536, False), (64, 1568, False), (64, 2080, False), (64, 3072, False),
    (64, 2048, True), (64, 2112, True), (64, 3072, True), (64, 3136, True),
    (64, 4096, True), (64, 5184, True), (64, 6144, True), (8192, 1024, True),
    (8224, 1024, True), (8224, 1088, True)])
def test_few_rows(m, n, k, fp8):
    """Products of 16 x 16 and, of more rows or odd lengths of sums, of 32 x 32, whole
    and in parts, of fewer columns of x than there are waves too."""
    torch.manual_seed(m + k)
    ws, scale, w = _weight(n, k, 0, fp8)
    x = torch.randn(m, k, device=DEV).bfloat16()
    e, ref = ops.ext(), x.double() @ w.t()
    args = (e.decode_swizzle_x(x), ws) + ((scale,) if fp8 else ()) + (m, n, k)
    y = (e.decode_gemm_fp8 if fp8 else e.decode_gemm)(*args)
    assert _rel(y, ref) < BF16
    raw = e.decode_gemm_fp8(*args, raw=True) if fp8 else \
        e.decode_gemm_raw(*args, True)
    if raw.dtype == torch.float32:
        assert _rel(raw.double().sum(0), ref) < 1e-5


@pytest.mark.parametrize("m", [1, 33, 64, 65, 128])
@pytest.mark.parametrize("inter,k", [(16, 1024), (10256, 1040)])
def test_gated_unit_of_rows(m, inter, k):
    torch.manual_seed(m + inter)
    ws, _, w = _weight(2 * inter, k, inter, False)
    x = (torch.randn(m, k, device=DEV) / k ** 0.5).bfloat16()
    y = x.double() @ w.t()
    ref = _act(y[:, :inter], False) * y[:, inter:]
    assert _rel(ops.ext().rows_glu(x, ws, 2 * inter, False), ref) < BF16


@pytest.mark.parametrize("m", [17, 64, 65])
@pytest.mark.parametrize("inter", [16384, 16400, 24576, 24592])
def test_wide_gated_unit_of_rows(m, inter):
    """Around the widths from where on a workgroup has two blocks of W and not four."""
    test_gated_unit_of_rows(m, inter, 1024)


@pytest.mark.parametrize("m", [48, 49, 64])
@pytest.mark.parametrize("inter,k", [(18432, 4096), (18432, 6656), (20480, 4096),
                                     (20480, 4128), (20496, 4096), (24576, 3408),
                                     (24576, 3424)])
def test_wide_gated_unit_of_long_rows(m, inter, k):
    """Around the sizes from where on more than 48 rows have four all the same."""
    test_gated_unit_of_rows(m, inter, k)


def _heads_case(m, hq, hkv, dh, vt):
    n, k = (hq + 2 * hkv) * dh, 1056
    cos, sin = ops.rope_tables(dh, 50, device=DEV)
    pos = torch.randint(0, 50, (m,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(16 * 10, device=DEV)[:m].to(torch.int32)
    if m > 2:
        slots[1] = -1               # written nowhere
    kc = torch.zeros(10, hkv, 16, dh, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros(10, hkv, *((dh, 16) if vt else (16, dh)), device=DEV,
                     dtype=torch.bfloat16)
    return n, k, cos, sin, pos, slots, kc, vc


def _heads_ref(y, cos, sin, pos, slots, kc, hq, hkv, dh):
    m = y.shape[0]
    y = y.view(m, hq + 2 * hkv, dh)
    c, s = (t.double()[pos.long()][:, None] for t in (cos, sin))
    a, b = y[:, :hq + hkv].split(dh // 2, -1)
    turned = torch.cat([a * c - b * s, b * c + a * s], -1)
    kr, vr = (torch.zeros(kc.shape, dtype=torch.float64, device=DEV)
              for _ in range(2))
    for i, t in enumerate(slots.tolist()):
        if t >= 0:
            kr[t // 16, :, t % 16] = turned[i, hq:]
            vr[t // 16, :, t % 16] = y[i, hq + hkv:]
    return turned[:, :hq], kr, vr, torch.cat([turned, y[:, hq + hkv:]], 1)


@pytest.mark.parametrize("m", [1, 16, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("hq,hkv,dh,vt", [(1, 1, 64, False), (4, 1, 128, True),
                                          (3, 3, 256, False),
                                          (48, 24, 128, False)])
@pytest.mark.parametrize("fp8", [False, True])
def test_heads(m, hq, hkv, dh, vt, fp8):
    if fp8 and m > 32:
        pytest.skip("8-bit weights are read by up to 32 rows")
    torch.manual_seed(m + dh)
    n, k, cos, sin, pos, slots, kc, vc = _heads_case(m, hq, hkv, dh, vt)
    ws, scale, w = _weight(n, k, dh // 2, fp8)
    x = torch.randn(m, k, device=DEV).bfloat16()
    e, y = ops.ext(), x.double() @ w.t()
    at = (cos, sin, pos, kc, vc, slots, hq)
    calls = []
    if m <= 32:
        xs, squares = e.decode_swizzle_x(x), _squares(x, 12)
        calls += [(1.0, lambda: e.decode_heads(xs, ws, scale, m, n, k, None,
                                               0.0, *at)),
                  (_inverse_rms(x), lambda: e.decode_heads(
                      xs, ws, scale, m, n, k, squares, 1e-5, *at))]
    if not fp8:
        calls += [(1.0, lambda: e.rows_heads(x, ws, n, *at)),
                  (1.0, lambda: e.rows_heads(x, ws, n, *at, rows=True))]
    for f, call in calls:
        kc.zero_(), vc.zero_()
        q, kr, vr, rows = _heads_ref(f * y, cos, sin, pos, slots, kc, hq, hkv,
                                     dh)
        got = call()
        assert _rel(got, q if got.dim() == 3 else rows.view(m, n)) < BF16
        assert _rel(kc, kr) < BF16
        assert _rel(vc.transpose(-1, -2) if vt else vc, vr) < BF16


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(64, 64), (64, 2080), (4096, 4096),
                                 (3072, 11008), (64, 3072), (64, 5632),
                                 (64, 6208), (64, 14336)])
@pytest.mark.parametrize("fp8", [False, True])
def test_residual_sum(m, n, k, fp8):
    e = ops.ext()
    if not e.decode_res_supported(m, n, k, fp8):
        assert fp8 and k % 64
        return
    torch.manual_seed(m + n)
    ws, scale, w = _weight(n, k, 0, fp8)
    x = (torch.randn(m, k, device=DEV) / k ** 0.5).bfloat16()
    res = torch.randn(m, n, device=DEV).bfloat16()
    g = torch.randn(n, device=DEV).bfloat16()
    ref = res.double() + x.double() @ w.t()
    for rows in (False, True):
        s, y, squares = e.decode_res(e.decode_swizzle_x(x), ws, scale, res, g,
                                     rows)
        assert _rel(s, ref) < BF16
        assert _rel(y if rows else _rows(y, n, m), ref * g.double()) < BF16
        assert squares.shape == (m, n // 16)
        assert _rel(squares.sum(1), ref.square().sum(1)) < 1e-4


@pytest.mark.parametrize("m", [1, 20, 32, 50, 128])
@pytest.mark.parametrize("fp8", [False, True])
def test_products_of_paired_copies(m, fp8):
    """A product that ends in nothing else gives its columns in their own
    order, whatever the order of the copy, and the same bits."""
    from runbooks_amd.ops.linear import (decode_linear_raw, fast_linear,
                                         quantize_fp8, register_decode_weight,
                                         rows_parts, wide_linear)
    torch.manual_seed(m)
    # sizes of each kernel: split or not, in rows or as an operand
    for n in (1536, 10752):
        w = torch.randn(n, 2048, device=DEV).bfloat16()
        x = torch.randn(m, 2048, device=DEV).bfloat16()
        products = [fast_linear, wide_linear]
        if m <= 32:
            products.append(lambda x, w: decode_linear_raw(x, w)[0])
        elif not fp8:
            products.append(rows_parts)
        got = []
        with torch.no_grad():
            for half in (0, 64, n // 2):
                (quantize_fp8 if fp8 else register_decode_weight)(w, half)
                got.append([p(x, w) for p in products])
        for paired in got[1:]:
            for a, b in zip(paired, got[0]):
                assert torch.equal(a, b)


def _model(kv, inter, hidden=1024, eight_bit=False, heads=8, dh=128,
           act="silu_glu"):
    from runbooks_amd.models import build_model, get_config
    from runbooks_amd.models.config import register
    from runbooks_amd.models.transformer import fuse_for_inference
    cfg = dataclasses.replace(
        get_config("smoke-llama"),
        name=f"ends-{kv}-{inter}-{hidden}-{heads}-{dh}-{act}",
        hidden_size=hidden, num_heads=heads, num_kv_heads=kv, head_dim=dh,
        intermediate_size=inter, num_layers=2, act=act)
    register(cfg)
    m = build_model(cfg.name, dtype=torch.bfloat16, tp=1, device=DEV, seed=3)
    return fuse_for_inference(m.eval(), load_in_8bit=eight_bit)


def _step(m, batch, fp8):
    """Arguments of a decode step behind caches of random contents."""
    g = torch.Generator(device=DEV).manual_seed(batch)
    caches = m.alloc_caches(batch * 2 + 1, DEV, fp8=fp8)
    for layer in caches:
        hkv, dh = layer[0].shape[1], layer[0].shape[3]
        k, v = (torch.randn(batch * 32, hkv, dh, device=DEV,
                            generator=g).bfloat16() for _ in range(2))
        ops.kv_append(k, v, *layer, torch.arange(batch * 32, device=DEV,
                                                 dtype=torch.int32))
    i32 = dict(dtype=torch.int32, device=DEV)
    lens = torch.arange(batch, **i32) % 31 + 1
    return (torch.arange(batch, device=DEV) % 50, lens - 1, caches,
            torch.arange(batch, **i32) * 32 + lens - 1,
            torch.arange(2 * batch, **i32).view(batch, 2), lens)


@pytest.mark.parametrize("batch", [1, 16, 17, 32])
@pytest.mark.parametrize("kv,inter,hidden,eight_bit", [
    (8, 2048, 1024, False), (2, 1040, 1024, False), (8, 6144, 1024, False),
    (8, 2048, 1024, True), (8, 2048, 4160, False)])
def test_decode_step(monkeypatch, batch, kv, inter, hidden, eight_bit):
    """A whole step on these kernels and on the modules: some twenty roundings
    of 2^-9 a layer, two layers, not in the same places."""
    from runbooks_amd.models import decode_chain
    from runbooks_amd.models.transformer import MLP, Attention, Block
    m = _model(kv, inter, hidden, eight_bit)
    args = _step(m, batch, eight_bit)
    with torch.no_grad():
        assert decode_chain.layers_of(m, Block, Attention, MLP) is not None
        got = m.decode(*args)
        monkeypatch.setattr(decode_chain, "layers_of", lambda *a: None)
        ref = m.decode(*args)
    assert _rel(got, ref.double()) < 2e-2


@pytest.mark.parametrize("batch", [16, 17, 24, 25, 32])
@pytest.mark.parametrize("inter,hidden,first", [
    (21488, 3072, 33), (21504, 3040, 33), (21504, 3072, 25), (28672, 3072, 25),
    (28688, 3072, 33), (21504, 5088, 25), (21504, 5120, 17), (16400, 3584, 25),
    (16400, 4096, 33), (16384, 3584, 17)])
def test_wide_gated_unit_of_a_step(monkeypatch, batch, inter, hidden, first):
    """As test_decode_step, around the sizes of wide gated units that take rows, from
    `first` on."""
    from runbooks_amd.models import decode_chain
    m = _model(8, inter, hidden)
    args = _step(m, batch, False)
    seen, plain = [], ops.ext().rows_glu

    def rows_glu(*a):
        seen.append(1)
        return plain(*a)
    with torch.no_grad():
        monkeypatch.setattr(ops.ext(), "rows_glu", rows_glu)
        got = m.decode(*args)
        assert len(seen) == (2 if batch >= first else 0)
        monkeypatch.setattr(decode_chain, "layers_of", lambda *a: None)
        ref = m.decode(*args)
    assert _rel(got, ref.double()) < 2e-2


@pytest.mark.parametrize("batch", [1, 16, 17, 32])
@pytest.mark.parametrize("kv,inter,hidden,fp8,few,many", [
    (8, 8192, 1024, False, 0, 0), (8, 8224, 1024, False, 0, 1),
    (2, 16384, 1024, False, 0, 1), (8, 16400, 1024, False, 1, 1),
    (8, 16400, 1024, True, 0, 0), (8, 5120, 4352, False, 3, 3)])
def test_sums_in_parts(monkeypatch, batch, kv, inter, hidden, fp8, few, many):
    """As test_decode_step, around the lengths from where on the sums of up to 16 and
    of more rows go in parts (`few` and `many` of two layers' four, the last of which
    is another kernel's), with wide residuals and ahead of 8-bit caches."""
    from runbooks_amd.models import decode_chain
    m = _model(kv, inter, hidden)
    args = _step(m, batch, fp8)
    seen, plain = [], ops.ext().parts_res

    def parts_res(*a):
        seen.append(1)
        return plain(*a)
    with torch.no_grad():
        monkeypatch.setattr(ops.ext(), "parts_res", parts_res)
        got = m.decode(*args)
        assert len(seen) == (few if batch <= 16 else many)
        monkeypatch.setattr(decode_chain, "layers_of", lambda *a: None)
        ref = m.decode(*args)
    assert _rel(got, ref.double()) < 2e-2


def test_hooked_modules_are_called():
    m = _model(8, 2048)
    args = _step(m, 3, False)
    seen = []
    with torch.no_grad():
        want = m.decode(*args)
        hook = m.blocks[1].mlp.register_forward_hook(
            lambda mod, x, y: seen.append(y))
        got = m.decode(*args)
        hook.remove()
    assert len(seen) == 1
    assert _rel(got, want.double()) < 2e-2


@pytest.mark.parametrize("which", ["attention", "block"])
def test_methods_of_an_object_are_called(which):
    """Decoding goes by the step of an attention or a block that has one of its
    own."""
    m = _model(8, 2048)
    args = _step(m, 3, False)
    seen = []
    blk = m.blocks[1]
    owner, name = (blk.attn, "forward_decode") if which == "attention" else \
        (blk, "forward_decode_fused")
    plain = getattr(owner, name)

    def step(*a, **kw):
        seen.append(1)
        return plain(*a, **kw)
    with torch.no_grad():
        want = m.decode(*args)
        setattr(owner, name, step)
        got = m.decode(*args)
    assert len(seen) == 1
    assert _rel(got, want.double()) < 2e-2


@pytest.mark.parametrize("batch", [33, 64, 65, 128])
@pytest.mark.parametrize("kv,inter", [(8, 2048), (2, 1040), (2, 12288)])
def test_wide_decode_step(monkeypatch, batch, kv, inter):
    """As test_decode_step, of more rows."""
    m = _model(kv, inter)
    args = _step(m, batch, False)
    with torch.no_grad():
        got = m.decode(*args)
        for name in ("rows_heads", "rows_glu", "rows_parts"):
            monkeypatch.setattr(ops, name, lambda *a, **k: None)
        ref = m.decode(*args)
    assert _rel(got, ref.double()) < 2e-2


@pytest.mark.parametrize("tokens", [31, 33, 128, 129])
@pytest.mark.parametrize("kv", [2, 8])
def test_short_prompt(monkeypatch, tokens, kv):
    """Logits and cached keys and values of a prompt on these kernels and on the
    modules; the bound as in test_decode_step."""
    m = _model(kv, 2048)
    i32 = dict(dtype=torch.int32, device=DEV)

    def prompt():
        caches = m.alloc_caches(16, DEV)
        with torch.no_grad():
            logits = m.prefill(torch.arange(tokens, device=DEV)[None] % 50,
                               torch.arange(tokens, **i32), caches,
                               torch.arange(tokens, **i32) + 5)
        return [logits] + [c for layer in caches for c in layer]

    got = prompt()
    for name in ("rows_heads", "rows_glu", "rows_parts"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    for a, b in zip(got, prompt()):
        assert _rel(a, b.double()) < 2e-2


@pytest.mark.parametrize("tokens", [1, 9, 16, 17, 32])
@pytest.mark.parametrize("kv,inter,eight_bit", [
    (8, 2048, False), (2, 1040, False), (2, 6144, False), (8, 2048, True)])
def test_shortest_prompts(monkeypatch, tokens, kv, inter, eight_bit):
    """Prompts of up to 32 tokens, whose products end in the rotation and the
    gated unit: as test_short_prompt, the products of modules called in their
    place."""
    m = _model(kv, inter, eight_bit=eight_bit)
    i32 = dict(dtype=torch.int32, device=DEV)
    ended = []

    def prompt():
        caches = m.alloc_caches(16, DEV)
        with torch.no_grad():
            logits = m.prefill(torch.arange(tokens, device=DEV)[None] % 50,
                               torch.arange(tokens, **i32), caches,
                               torch.arange(tokens, **i32) + 5)
        return [logits] + [c for layer in caches for c in layer]

    for name in ("rows_heads", "few_rows_mlp"):
        def seen(*a, f=getattr(ops, name), **k):
            y = f(*a, **k)
            ended.append(y is not None)
            return y
        monkeypatch.setattr(ops, name, seen)
    got = prompt()
    # 8-bit weights have their own product of q, k and v
    assert ended == [not eight_bit, True] * 2
    for name in ("rows_heads", "few_rows_mlp"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    for a, b in zip(got, prompt()):
        assert _rel(a, b.double()) < 2e-2


@pytest.mark.parametrize("m", [33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(32, 1024), (1024, 1088), (4096, 8192)])
def test_residual_sum_of_rows(m, n, k):
    x = torch.randn(m, k, device=DEV).bfloat16()
    res = (torch.randn(m, n, device=DEV) * k ** 0.5).bfloat16()
    gamma = torch.randn(n, device=DEV).bfloat16()
    ws, _, w = _weight(n, k, 0, False)
    assert ops.ext().rows_res_supported(m, n, k)
    out, y, squares = ops.ext().rows_res(x, ws, res, gamma)
    want = res.double() + x.double() @ w.t()
    assert _rel(out, want) < BF16
    assert _rel(y, want * gamma.double()) < BF16
    assert _rel(squares.sum(1), want.square().sum(1)) < 1e-5


@pytest.mark.parametrize("m,n,k", [(16, 1024, 1024), (32, 1024, 1024),
                                   (65, 1024, 1024),
                                   (48, 1040, 1024), (48, 1024, 1056),
                                   (48, 4128, 1024)])
def test_refused_residual_sums_of_rows(m, n, k):
    assert not ops.ext().rows_res_supported(m, n, k)
    x = torch.zeros(m, k, device=DEV).bfloat16()
    res = torch.zeros(m, n, device=DEV).bfloat16()
    ws = torch.zeros(n * k, device=DEV).bfloat16()
    with pytest.raises(RuntimeError):
        ops.ext().rows_res(x, ws, res, res[0])


@pytest.mark.parametrize("m", [33, 64])
@pytest.mark.parametrize("parts,n", [(2, 1280), (4, 4096), (8, 8192)])
def test_residual_of_parts(m, parts, n):
    """Sums of parts and residual with the norm's squares, fp32 throughout."""
    assert ops.ext().parts_res_supported(n)
    p = torch.randn(parts, m, n, device=DEV)
    res = torch.randn(m, n, device=DEV).bfloat16()
    gamma = torch.randn(n, device=DEV).bfloat16()
    out, y, squares = ops.ext().parts_res(p, res, gamma)
    want = res.double() + p.double().sum(0)
    assert _rel(out, want) < BF16
    assert _rel(y, want * gamma.double()) < BF16
    assert _rel(squares.sum(1), want.square().sum(1)) < 1e-5


@pytest.mark.parametrize("m", [33, 48, 64])
@pytest.mark.parametrize("inter,k,parts", [(2048, 1024, 4), (5504, 4096, 128),
                                           (2064, 1056, 256)])
def test_units_of_rows_normed_late(m, inter, k, parts):
    """rows_glu and rows_heads of 33 to 64 rows that still lack their 1 / rms."""
    x = torch.randn(m, k, device=DEV).bfloat16()
    squares = _squares(x, parts)
    w = (torch.randn(2 * inter, k, device=DEV) / k ** 0.5).bfloat16()
    ws = ops.ext().decode_swizzle_w(w, inter)
    both = (x.double() * _inverse_rms(x)) @ w.double().t()
    want = _act(both[:, :inter], False) * both[:, inter:]
    h = ops.ext().rows_glu(x, ws, 2 * inter, False, False, squares, 1e-5)
    assert _rel(h, want) < BF16

    dh, hq, hkv = 128, 16, 4
    n = (hq + 2 * hkv) * dh
    w = torch.randn(n, k, device=DEV).bfloat16()
    ws = ops.ext().decode_swizzle_w(w, dh // 2)
    i32 = dict(dtype=torch.int32, device=DEV)
    kc = torch.zeros(8, hkv, 16, dh, device=DEV).bfloat16()
    vc = torch.zeros_like(kc)
    ones = torch.ones(8, dh // 2, device=DEV)
    y = ops.ext().rows_heads(x, ws, n, ones, ones * 0, torch.zeros(m, **i32),
                             kc, vc, torch.arange(m, **i32), hq, True, squares,
                             1e-5)
    want = (x.double() * _inverse_rms(x)) @ w.double().t()
    assert _rel(y.reshape(m, -1), want) < BF16


def _served_by_rows(monkeypatch):
    """Blocks that run_rows took, call by call."""
    from runbooks_amd.models import decode_chain
    seen, plain = [], decode_chain.run_rows

    def run(*args):
        out = plain(*args)
        seen.append(out[2])
        return out
    monkeypatch.setattr(decode_chain, "run_rows", run)
    return seen


@pytest.mark.parametrize("tokens", [33, 48, 64])
@pytest.mark.parametrize("kv,inter,hidden", [(8, 2048, 1024), (2, 6144, 1024),
                                             (8, 12288, 1024), (8, 2048, 4096)])
@pytest.mark.parametrize("decode", [False, True])
def test_steps_of_rows(monkeypatch, tokens, kv, inter, hidden, decode):
    """A prompt and a step of 33 to 64 rows on these kernels and on the modules,
    bound as in test_decode_step, and with a hook on the second block, which is
    called in its place and gets the first one's result."""
    m = _model(kv, inter, hidden)
    i32 = dict(dtype=torch.int32, device=DEV)
    seen = _served_by_rows(monkeypatch)

    def step():
        if decode:
            args = _step(m, tokens, False)
            caches = args[2]
        else:
            caches = m.alloc_caches(16, DEV)
            args = (torch.arange(tokens, device=DEV)[None] % 50,
                    torch.arange(tokens, **i32), caches,
                    torch.arange(tokens, **i32) + 5)
        with torch.no_grad():
            logits = m.decode(*args) if decode else m.prefill(*args)
        return [logits] + [c for layer in caches for c in layer]

    got = step()
    called = []
    hook = m.blocks[1].mlp.register_forward_hook(
        lambda mod, x, y: called.append(y.shape))
    mixed = step()
    hook.remove()
    monkeypatch.setattr(type(m), "_few_rows",
                        lambda self, x, *a: self._blocks(x, a[-1]))
    ref = step()
    assert seen == [2, 1] and len(called) == 1
    for a, b, c in zip(got, mixed, ref):
        assert _rel(a, c.double()) < 2e-2 and _rel(b, c.double()) < 2e-2


@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("why", ["hook", "copy", "norm"])
def test_rows_handed_over(monkeypatch, decode, why):
    """What run_rows leaves to the modules, of a block whose MLP has a hook, one
    whose copy is older than its weight, and one whose norm has a hook: to a norm
    that adds them up, the last product's sums in fp32 parts, unrounded."""
    from runbooks_amd.models import decode_chain
    m = _model(8, 2048)
    i32 = dict(dtype=torch.int32, device=DEV)
    if decode:
        args = _step(m, 40, False)
    else:
        args = (torch.arange(40, device=DEV)[None], torch.arange(40, **i32),
                m.alloc_caches(16, DEV), torch.arange(40, **i32))
    blk = m.blocks[1]
    if why == "hook":
        blk.mlp.register_forward_hook(lambda *a: None)
    elif why == "copy":
        with torch.no_grad():
            blk.mlp.down_proj.weight.mul_(0.5)
    else:
        blk.norm2.register_forward_hook(lambda *a: None)
    seen, given = [], []
    run, product = decode_chain.run_rows, ops.ext().decode_gemm_rows

    def run_rows(*a):
        monkeypatch.setattr(ops.ext(), "decode_gemm_rows", lambda x, *b:
                            given.append(x) or product(x, *b))
        seen.append(run(*a))
        monkeypatch.setattr(ops.ext(), "decode_gemm_rows", product)
        return seen[-1]
    monkeypatch.setattr(decode_chain, "run_rows", run_rows)
    with torch.no_grad():
        (m.decode if decode else m.prefill)(*args)
    _, delta, blocks = seen[0]
    assert blocks == 1
    want = given[-1].double() @ m.blocks[0].mlp.down_proj.weight.double().t()
    if why == "norm":           # adds no parts up
        assert delta.dtype == torch.bfloat16 and _rel(delta, want) < BF16
    else:
        assert delta.dtype == torch.float32 and delta.shape[1:] == want.shape
        assert _rel(delta.sum(0), want) < 1e-5


@pytest.mark.parametrize("rows", ["step", "prompt", "prompts"])
@pytest.mark.parametrize("stale", [False, True])
@pytest.mark.parametrize("kv,inter,hidden,heads,dh,act", [
    (8, 2048, 1024, 8, 128, "gelu_glu"), (4, 2048, 1024, 16, 64, "silu_glu"),
    (4, 2048, 1024, 4, 256, "gelu_glu"),
    (2, 1024, 8448, 8, 128, "silu_glu")])       # a down projection in one part
def test_rows_of_other_models(monkeypatch, rows, stale, kv, inter, hidden, heads,
                              dh, act):
    """As test_steps_of_rows: units of GELU, heads of 64 and 256, sums that no
    kernel takes in parts, two prompts at once, and a second block whose copies
    are older than its weights."""
    m = _model(kv, inter, hidden, heads=heads, dh=dh, act=act)
    i32 = dict(dtype=torch.int32, device=DEV)
    seen = _served_by_rows(monkeypatch)
    if stale:
        with torch.no_grad():
            m.blocks[1].mlp._gateup_w.mul_(0.5)

    def step():
        if rows == "step":
            args = _step(m, 40, False)
            caches = args[2]
        else:
            caches = m.alloc_caches(16, DEV)
            n, of = (2, 24) if rows == "prompts" else (1, 47)
            args = (torch.arange(n * of, device=DEV).view(n, of) % 50,
                    torch.arange(of, **i32).repeat(n), caches,
                    torch.arange(n * of, **i32) + 5)
        with torch.no_grad():
            logits = (m.decode if rows == "step" else m.prefill)(*args)
        return [logits] + [c for layer in caches for c in layer]

    got = step()
    monkeypatch.setattr(type(m), "_few_rows",
                        lambda self, x, *a: self._blocks(x, a[-1]))
    assert seen == [1 if stale else 2]
    for a, b in zip(got, step()):
        assert _rel(a, b.double()) < 2e-2
