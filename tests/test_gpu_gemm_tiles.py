"""Products in tiles (csrc/gemm_tiles.hip) at the edges of their tiles, with
their sums in parts and ended by a gated unit, against fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = range(7)        # 256x256 192x256 256x192 256x128 128x256 128x192 128x128


def _inputs(m, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) * k ** -0.5).bfloat16()
    return x, w


def _check(got, x, w, rounding):
    """Sums of k products in fp32, in any order: off by at most k eps times the
    sum of their absolute values; and their rounding."""
    ref = x.float() @ w.float().t()
    size = x.float().abs() @ w.float().abs().t()
    bound = rounding * ref.abs() + 2 * x.shape[1] * 2.0 ** -24 * size
    assert bool(((got.float() - ref).abs() <= bound).all())


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [
    (1, 4, 256),            # less than a fragment, the fewest columns of K
    (129, 260, 320),        # remainders of every tile, odd K-tiles
    (256, 512, 512),        # whole tiles
    (513, 1028, 448),
    (4100, 4360, 256),      # several tiles for a workgroup
])
def test_product(tile, m, n, k):
    from runbooks_amd import ops
    x, w = _inputs(m, n, k)
    _check(ops.ext().tile_gemm(x, w, tile=tile), x, w, 2.0 ** -8)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k,parts", [
    (129, 260, 1088, 4),    # 5, 5, 5 and 2 K-tiles are not enough: refused
    (130, 516, 1024, 4),
    (300, 260, 576, 2),     # 5 and 4
    (257, 4100, 1472, 3),
])
def test_parts(tile, m, n, k, parts):
    from runbooks_amd import ops
    x, w = _inputs(m, n, k)
    run = lambda: ops.ext().tile_gemm(x, w, parts, tile=tile, parts=parts)  # noqa: E731
    if -(-(k // 64) // parts) * (parts - 1) + 4 > k // 64:
        with pytest.raises(RuntimeError):
            run()
        return
    y = run()
    assert y.shape == (parts, m, n) and y.dtype == torch.float32
    _check(y.sum(0), x, w, 2.0 ** -22)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("glu", [1, 2])
@pytest.mark.parametrize("m,n,k", [(1, 8, 256), (200, 520, 320),
                                   (4100, 4360, 256)])
def test_gated_unit(tile, glu, m, n, k):
    from runbooks_amd import ops
    x, w = _inputs(m, n, k)
    got = ops.ext().tile_gemm(x, w, glu=glu, tile=tile).float()
    g, u = (x.float() @ w.float().t()).chunk(2, 1)
    act = torch.nn.functional.silu(g) if glu == 1 else \
        torch.nn.functional.gelu(g, approximate="tanh")
    ref = act * u
    # the product's errors (of values around 1, 1e-5) through gate and unit,
    # and one rounding
    assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all())


@pytest.mark.parametrize("tile", [-1, *TILES])
@pytest.mark.parametrize("m,widths,k", [
    (1, [16], 256), (300, [208, 16, 64], 320),  # siblings within a tile
    (513, [512, 576], 448), (4100, [2048, 1152, 1152], 256)])
def test_adapters(tile, m, widths, k):
    from runbooks_amd import ops
    x, w = _inputs(m, sum(widths), k)
    t = torch.randn(len(widths), m, 16, device="cuda").bfloat16()
    bs = [torch.randn(n, 16, device="cuda").bfloat16() for n in widths]
    got = ops.ext().tile_lora(x, w, t, bs, 0.3, tile=tile)
    more = torch.cat([ti.float() @ b.float().t() for ti, b in zip(t, bs)], 1)
    ref = x.float() @ w.float().t() + 0.3 * more
    # sums of k products of size 1 / sqrt(k) and of 16 of size 1
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -24 * (2 * k ** 1.5 + 2 * 16 * 16)
    assert bool(((got.float() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k", [(700, 22016, 4096), (2200, 22016, 1024),
                                   (1800, 28680, 1024)])
def test_two_launches(m, n, k):
    """Sizes of more tiles than whole rounds: columns in tiles of two sizes."""
    from runbooks_amd import ops
    _, parts, rest, split = ops.ext().tile_gemm_choice(m, n, k)
    assert parts == 1 and rest >= 0 and 0 < split < n
    x, w = _inputs(m, n, k)
    _check(ops.ext().tile_gemm(x, w), x, w, 2.0 ** -8)
    g, u = (x.float() @ w.float().t()).chunk(2, 1)
    ref = torch.nn.functional.silu(g) * u
    got = ops.ext().tile_gemm(x, w, glu=1).float()
    assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all())


def _with_adapters(x, w, t, bs, scale):
    more = torch.cat([ti.float() @ b.float().t() for ti, b in zip(t, bs)], 1)
    return x.float() @ w.float().t() + scale * more


@pytest.mark.parametrize("m,widths,k", [
    (700, [11008, 11008], 4096),            # siblings meet in the first launch
    (700, [18432, 2560, 1024], 4096),       # in the second one
    (3001, [4096, 1024, 1024], 4096)])      # between them, and in the second
def test_adapters_in_two_launches(m, widths, k):
    from runbooks_amd import ops
    n = sum(widths)
    _, _, rest, split = ops.ext().tile_gemm_choice(m, n, k)
    assert rest >= 0 and 0 < split < n
    x, w = _inputs(m, n, k)
    t = torch.randn(len(widths), m, 16, device="cuda").bfloat16()
    bs = [torch.randn(c, 16, device="cuda").bfloat16() for c in widths]
    got = ops.ext().tile_lora(x, w, t, bs, 0.3)
    ref = _with_adapters(x, w, t, bs, 0.3)
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -24 * (2 * k ** 1.5 + 2 * 16 * 16)
    assert bool(((got.float() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,widths,k,tiles", [
    (1100, [2048], 256, True), (129, [4096, 1024, 1024], 320, True),
    (1100, [4096], 8192, False), (512, [4096], 256, False)])
def test_products_with_adapters(monkeypatch, m, widths, k, tiles):
    """Both ways that wide_product_lora may take, by its own rule and against
    it: the library's rounds the product and the sum."""
    from runbooks_amd import ops
    from runbooks_amd.ops import linear
    n = sum(widths)
    x, w = _inputs(m, n, k)
    t = torch.randn(len(widths), m, 16, device="cuda").bfloat16()
    bs = [torch.randn(c, 16, device="cuda").bfloat16() for c in widths]
    ref = _with_adapters(x, w, t, bs, 0.3)
    tile = ops.ext().tile_lora(x, w, t, bs, 0.3)
    got = linear.wide_product_lora(x, w, t, bs, 0.3)
    assert linear._lora_in_tiles(m, n, k) is tiles
    assert torch.equal(got, tile) is tiles
    monkeypatch.setattr(linear, "_lora_in_tiles", lambda *a: not tiles)
    other = linear.wide_product_lora(x, w, t, bs, 0.3)
    sums = 2.0 ** -24 * (2 * k ** 1.5 + 2 * 16 * 16)
    product = (x.float() @ w.float().t()).abs()
    for y in (got, other):
        bound = 2.0 ** -8 * (ref.abs() + product * 1.01) + sums
        assert bool(((y.float() - ref).abs() <= bound).all())


def test_packed_adapter_in_tiles():
    """A LoRA layer whose product ends with its adapter, forward and backward,
    against fp32: results and gradients of one bf16 rounding and fp32 sums over
    inputs of one rounding more (t, dt, the gradients' own)."""
    from torch import nn

    from runbooks_amd.ops import linear
    from runbooks_amd.train.lora import LoRALinear
    m, n, k = 1100, 2048, 512
    assert linear._lora_in_tiles(m, n, k)
    torch.manual_seed(0)
    base = nn.Linear(k, n, bias=False, device="cuda", dtype=torch.bfloat16)
    base.weight.requires_grad_(False)
    layer = LoRALinear(base, r=16, alpha=32, dtype=torch.bfloat16).cuda()
    with torch.no_grad():
        layer.lora_a.normal_(0, k ** -0.5)
        layer.lora_b.normal_(0, 0.25)
    x = torch.randn(m, k, device="cuda").bfloat16().requires_grad_()
    dy = torch.randn(m, n, device="cuda").bfloat16()
    y = layer(x)
    assert y.grad_fn.name() == "_LoRAPackedBackward"
    y.backward(dy)
    leaves = [v.detach().float().requires_grad_()
              for v in (x, layer.lora_a, layer.lora_b)]
    xf, a, b = leaves
    ref = xf @ base.weight.float().t() + layer.scale * (xf @ a.t()) @ b.t()
    ref.backward(dy.float())
    for got, want in ((y, ref), (x.grad, xf.grad), (layer.lora_a.grad, a.grad),
                      (layer.lora_b.grad, b.grad)):
        assert float((got - want).detach().norm() / want.detach().norm()) < 2 * 2.0 ** -8


@pytest.mark.parametrize("m,n,k,taken", [
    (1000, 8192, 8256, True), (1793, 4096, 8256, True),
    (1000, 8192, 8192, False), (1700, 3072, 8256, False)])
def test_one_round_of_tiles(m, n, k, taken):
    """Long rows that one round of tiles does, and their neighbours."""
    from runbooks_amd import ops
    from runbooks_amd.ops import linear
    x, w = _inputs(m, n, k)
    y = linear._one_round(x, w)
    assert (y is not None) is taken
    got = linear.wide_product(x, w)
    _check(got, x, w, 2.0 ** -8)
    if taken:
        assert torch.equal(got, ops.ext().tile_gemm(x, w))


@pytest.mark.parametrize("m,n,k,taken", [
    (129, 12288, 256, True), (256, 18432, 320, True), (320, 12288, 2048, True),
    (257, 12288, 1024, False), (256, 20480, 256, False)])
def test_wide_products_of_few_rows(monkeypatch, m, n, k, taken):
    from runbooks_amd import ops
    from runbooks_amd.ops import linear
    x, w = _inputs(m, n, k)
    called = []
    monkeypatch.setattr(linear, "fast_linear",
                        lambda *a, f=linear.fast_linear: called.append(1) or
                        f(*a))
    with torch.no_grad():
        got = ops.wide_linear(x, w)
    _check(got, x, w, 2.0 ** -8)
    assert (not called) is taken


@pytest.mark.parametrize("m,n,k,parts", [
    (129, 4096, 4096, 4), (512, 4096, 11008, 4), (300, 3072, 24576, 3),
    (1793, 4096, 11008, 1),                     # whole, in one round
    (768, 4096, 4096, None), (400, 2048, 2048, None)])
def test_sums_for_the_norm(m, n, k, parts):
    """rows_parts of more than 128 rows: parts, one round of tiles, or None
    where the library is as fast; refused are rows and parameters that do not
    lie as the kernel reads them."""
    from runbooks_amd import ops
    x, w = _inputs(m, n, k)
    with torch.no_grad():
        y = ops.rows_parts(x, w)
        assert (None if y is None else
                y.shape[0] if y.dim() == 3 else 1) == parts
        if y is not None:
            _check(y.sum(0) if y.dim() == 3 else y, x, w, 2.0 ** -8)
        wide = torch.zeros(m, 2 * k, device="cuda", dtype=torch.bfloat16)
        assert ops.rows_parts(wide[:, :k], w) is None
        assert ops.rows_glu(x.float(), w.float(), False) is None
    assert ops.rows_parts(x, w) is None         # would be differentiated


def _down_inputs(m, n, k, siblings, apart=False):
    """x [m, k], W [k, n], t and A of siblings, one after the other in memory
    or, `apart`, further from each other than 2 GiB."""
    x, w = _inputs(m, n, k)
    t = torch.randn(siblings, m, 16, device="cuda").bfloat16()
    if apart:
        room = torch.empty((1 << 30) + 4 * 16 * n, device="cuda",
                           dtype=torch.bfloat16)
        As = [room[-16 * n:].view(16, n), room[:16 * n].view(16, n)][:siblings]
        for a in As:
            a.normal_()
    else:
        As = [torch.randn(16, n, device="cuda").bfloat16()
              for _ in range(siblings)]
    return x, w.t().contiguous(), t, As


def _check_down(got, x, w, t, As, rounding):
    """fp32 sums of k + 16 n products in any order, and their rounding."""
    ref = x.double() @ w.double()
    size = x.abs().double() @ w.abs().double()
    for ti, a in zip(t, As):
        ref += ti.double() @ a.double()
        size += ti.abs().double() @ a.abs().double()
    bound = rounding * ref.abs() + \
        2 * (x.shape[1] + 16 * len(As)) * 2.0 ** -24 * size
    assert bool(((got.double() - ref).abs() <= bound).all())


DOWN_TILES = [0, 1, 3, 4, 6]            # of 128 and 256 columns


@pytest.mark.parametrize("tile", DOWN_TILES)
@pytest.mark.parametrize("m,n,k,siblings", [
    (1, 8, 256, 0),             # less than a fragment, the fewest rows of W
    (129, 264, 320, 1),         # remainders of every tile, odd K-tiles
    (256, 512, 512, 2),         # whole tiles
    (513, 1032, 448, 3),
    (4100, 4360, 256, 3)])      # several tiles for a workgroup
def test_product_down_columns(tile, m, n, k, siblings):
    from runbooks_amd import ops
    args = _down_inputs(m, n, k, siblings)
    _check_down(ops.ext().tile_gemm_down(*args, tile=tile), *args, 2.0 ** -8)


@pytest.mark.parametrize("tile", DOWN_TILES)
@pytest.mark.parametrize("m,n,k,siblings,parts", [
    (130, 520, 1024, 1, 4), (300, 264, 576, 3, 2), (257, 4104, 1472, 0, 3)])
def test_parts_down_columns(tile, m, n, k, siblings, parts):
    """The adapters go with the last part, once."""
    from runbooks_amd import ops
    args = _down_inputs(m, n, k, siblings)
    y = ops.ext().tile_gemm_down(*args, max_parts=parts, tile=tile, parts=parts)
    assert y.shape == (parts, m, n) and y.dtype == torch.float32
    _check_down(y.double().sum(0), *args, 2.0 ** -24)


def test_adapters_apart_in_memory():
    from runbooks_amd import ops
    args = _down_inputs(200, 512, 256, 2, apart=True)
    _check_down(ops.ext().tile_gemm_down(*args), *args, 2.0 ** -8)


def test_two_launches_down_columns():
    from runbooks_amd import ops
    m, n, k = 3001, 14336, 4096
    _, parts, rest, split = ops.ext().tile_gemm_down_choice(m, n, k, 4)
    assert parts == 1 and rest >= 0 and 0 < split < n
    args = _down_inputs(m, n, k, 1)
    _check_down(ops.ext().tile_gemm_down(*args), *args, 2.0 ** -8)


def test_infinite_values_stay_in_their_row_and_column():
    """Absent siblings and columns past the end are zeros times zeros."""
    from runbooks_amd import ops
    x, w, t, As = _down_inputs(300, 520, 512, 1)
    clean = ops.ext().tile_gemm_down(x, w, t, As)
    t[0, 7, 3] = float("inf")
    As[0][5, 11] = float("-inf")
    w[:, 519] = float("nan")
    got = ops.ext().tile_gemm_down(x, w, t, As)
    rows = [i for i in range(300) if i != 7]
    cols = [i for i in range(519) if i != 11]
    assert torch.equal(got[rows][:, cols], clean[rows][:, cols])
    assert not bool(got[:, 11].isfinite().any() | got[7, :519].isfinite().any())
    assert bool(got[:, 519].isnan().all())


@pytest.mark.parametrize("m,n,k,siblings,tiles", [
    (2048, 4096, 1024, 1, True), (300, 4096, 6144, 3, True),
    (1100, 4096, 4096, 1, False), (77, 64, 192, 2, False)])
def test_gradients_of_inputs(monkeypatch, m, n, k, siblings, tiles):
    """Both ways that wide_product_grad may take, by its own rule and, where
    the tiles take it, against it: the library's rounds the product and the
    sum."""
    from runbooks_amd import ops
    from runbooks_amd.ops import linear
    x, w, t, As = _down_inputs(m, n, k, siblings)
    ext = ops.ext()
    taken = ext.tile_gemm_down_takes(x, w)
    assert (taken and ext.tile_gemm_down_pays(m, n, k)) is tiles
    called = []
    monkeypatch.setattr(linear, "_library_grad",
                        lambda *a, f=linear._library_grad: called.append(1) or
                        f(*a))
    got = linear.wide_product_grad(x, w, t, As)
    assert (not called) is tiles
    other = ext.tile_gemm_down(x, w, t, As) if taken and not tiles else \
        linear._library_grad(x, w)
    if tiles or not taken:
        ext.lora_add_(other, t, As, 1.0, True)
    own, library = (got, other) if tiles else (other, got)
    if taken:
        _check_down(own, x, w, t, As, 2.0 ** -8)
    # the product's rounding, of whatever size it is, and the sum's
    ref = x.double() @ w.double()
    product = 2.0 ** -8 * ref.abs()
    ref = ref + sum(ti.double() @ a.double() for ti, a in zip(t, As))
    bound = 2.0 ** -8 * ref.abs() + product + 1e-4
    assert bool(((library.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("change", ["rows", "columns", "aligned", "type", "rank"])
def test_refused_down_columns(change):
    from runbooks_amd import ops
    x, w, t, As = _down_inputs(200, 512, 320, 1)
    if change == "rows":
        x, w = x[:, :300].contiguous(), w[:300]
    elif change == "columns":
        w = w[:, :508].contiguous()
    elif change == "aligned":
        x = torch.zeros(200 * 320 + 1, device="cuda",
                        dtype=torch.bfloat16)[1:].view(200, 320)
    elif change == "type":
        x, w = x.float(), w.float()
    else:
        t = t[:, :, :8].contiguous()
    assert ops.ext().tile_gemm_down_takes(x, w) is (change == "rank")
    with pytest.raises(RuntimeError):
        ops.ext().tile_gemm_down(x, w, t, As)


def test_one_row_does_not_reach_others():
    """An infinite and a NaN row stay to themselves."""
    from runbooks_amd import ops
    x, w = _inputs(300, 520, 512)
    clean = ops.ext().tile_gemm(x, w)
    x[7] = float("inf")
    x[299, 3] = float("nan")
    got = ops.ext().tile_gemm(x, w)
    keep = [i for i in range(300) if i not in (7, 299)]
    assert torch.equal(got[keep], clean[keep])
    assert bool(got[299].isnan().all()) and not bool(got[7].isfinite().any())


def test_parts_are_not_differentiated():
    """A norm's sum of parts is refused where its gradient would be lost."""
    from runbooks_amd import ops
    x = torch.randn(200, 64, device="cuda").bfloat16()
    parts = torch.randn(2, 200, 64, device="cuda")
    w = torch.ones(64, device="cuda").bfloat16()
    with pytest.raises(RuntimeError):
        ops.rmsnorm_res(x, parts, w, 1e-5)
    with torch.no_grad():
        s, _ = ops.rmsnorm_res(x, parts, w, 1e-5)
    ref = x.float() + parts.sum(0)
    # one rounding, and the order of three fp32 terms of up to 5
    assert bool(((s.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("n", [8, 24, 264, 1048])
def test_stores_of_eight_columns(tile, n):
    """Rows of whole pieces of 16 bytes that end within a pair of 16 x 16 results,
    and behind the first of one: y and its unit."""
    from runbooks_amd import ops
    x, w = _inputs(131, 2 * n, 320)
    _check(ops.ext().tile_gemm(x, w[:n].contiguous(), tile=tile), x, w[:n],
           2.0 ** -8)
    g, u = (x.float() @ w.float().t()).chunk(2, 1)
    ref = torch.nn.functional.silu(g) * u
    got = ops.ext().tile_gemm(x, w, glu=1, tile=tile).float()
    assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all())


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("widths", [[48], [16, 32], [208, 16, 48]])
def test_adapters_of_odd_results(tile, widths):
    """An odd number of 16 x 16 results, and siblings that meet within a pair."""
    from runbooks_amd import ops
    x, w = _inputs(131, sum(widths), 320)
    t = torch.randn(len(widths), 131, 16, device="cuda").bfloat16()
    bs = [torch.randn(n, 16, device="cuda").bfloat16() for n in widths]
    got = ops.ext().tile_lora(x, w, t, bs, 0.3, tile=tile)
    ref = _with_adapters(x, w, t, bs, 0.3)
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -24 * (2 * 320 ** 1.5 + 2 * 16 * 16)
    assert bool(((got.float() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k,tiles", [
    (321, 8192, 4096, False), (512, 6144, 4096, False), (900, 4096, 4096, True),
    (513, 3328, 256, False), (1030, 2052, 2048, True), (1400, 20484, 512, False),
    (1400, 4096, 8256, False),
    (400, 8196, 4096, True),        # no multiple of 256
    (1280, 4096, 2560, False), (2048, 3072, 2560, True),    # CUs idle, and not
    (2048, 8192, 1024, False), (1900, 11004, 512, True),    # whole rounds, short
    (2816, 6144, 1024, True), (2816, 6144, 6208, False),    # more rounds
    (10300, 256, 1024, True), (16384, 252, 512, False), (24600, 256, 256, False)])
def test_wide_products(monkeypatch, m, n, k, tiles):
    """wide_linear and wide_product go by the rule for tiles, on either side."""
    from runbooks_amd import ops
    from runbooks_amd.ops import linear
    x, w = _inputs(m, n, k)
    assert linear._many_in_tiles(m, n, k) is tiles
    called, tile_gemm = [], ops.ext().tile_gemm
    monkeypatch.setattr(ops.ext(), "tile_gemm",
                        lambda *a, **kw: called.append(1) or tile_gemm(*a, **kw))
    with torch.no_grad():
        for i, product in enumerate((ops.wide_linear, linear.wide_product), 1):
            _check(product(x, w), x, w, 2.0 ** -8)
            assert len(called) == (i if tiles else 0)


@pytest.mark.parametrize("m,n,k,tiles", [
    (3001, 20480, 256, True), (9800, 6144, 320, True), (2900, 20480, 256, False),
    (9800, 6140, 256, False), (3001, 20480, 5184, False)])
def test_large_products_with_adapters(m, n, k, tiles):
    from runbooks_amd.ops import linear
    assert linear._large_lora_in_tiles(m, n, k) is \
        (tiles and not linear._lora_in_tiles(m, n, k))
    if not tiles:
        return
    x, w = _inputs(m, n, k)
    t = torch.randn(1, m, 16, device="cuda").bfloat16()
    bs = [torch.randn(n, 16, device="cuda").bfloat16()]
    ref = _with_adapters(x, w, t, bs, 0.3)
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -24 * (2 * k ** 1.5 + 2 * 16 * 16)
    got = linear.wide_product_lora(x, w, t, bs, 0.3)
    assert bool(((got.float() - ref).abs() <= bound).all())
