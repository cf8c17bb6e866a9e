"""Products of layer-norm models' decode with the norm before and the residual or
the cache behind them (csrc/decode_affine.hip)."""
import pytest
import torch

from runbooks_amd import ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# one rounding to bf16 (half a unit of 8 bits) beside fp32 sums
BF16 = 2 ** -8 + 1e-4
ACTS = [lambda y: y, torch.relu, torch.nn.functional.gelu,
        lambda y: torch.nn.functional.gelu(y, approximate="tanh")]


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _normed(res, g, b, eps):
    x = res.double() - res.double().mean(1, keepdim=True)
    x = x * (x.square().mean(1, keepdim=True) + eps).rsqrt()
    return x * g.double() + b.double()


def _param(*shape):
    return torch.randn(*shape, device=DEV).bfloat16()


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 16, 17, 24])
@pytest.mark.parametrize("widths,k,act", [
    ([32], 32, 0), ([64, 32, 96], 96, 0), ([2080], 544, 2), ([3072], 768, 1),
    ([768, 768, 768], 768, 0), ([96], 1024, 3)])
def test_normed_products(m, widths, k, act):
    """The norm's result is rounded to bf16 (2^-9 of it each, which the sums
    average), then the product's."""
    e = ops.ext()
    if not e.normed_affine_supported(m, k):
        assert m * k > 24576
        return
    torch.manual_seed(m + k)
    res = torch.randn(m, k, device=DEV) * 3 + torch.randn(m, 1, device=DEV) * 5
    g, b = _param(k), _param(k)
    ws = [_param(n, k) for n in widths]
    bs = [_param(n) if i != 1 else None for i, n in enumerate(widths)]
    got = e.normed_affine(res, g, b, 1e-5, ws, bs, act)
    x = _normed(res, g, b, 1e-5)
    for y, w, c in zip(got, ws, bs):
        ref = x @ w.double().t()
        ref = ACTS[act](ref if c is None else ref + c.double())
        assert _rel(y, ref) < 2 * BF16
    if len(widths) == 1 and not e.affine_in_rows(m):
        h = e.normed_affine(res, g, b, 1e-5, ws, bs, act, True)[0]
        assert torch.equal(h.view(-1, 2, 32, 8)[:, :, :m].permute(2, 0, 1, 3)
                           .reshape(m, -1), got[0])


@pytest.mark.parametrize("m", [1, 4, 5, 24])
@pytest.mark.parametrize("heads,dh,vt", [(1, 32, False), (6, 64, False),
                                         (2, 128, True)])
def test_cached_keys_and_values(m, heads, dh, vt):
    e = ops.ext()
    torch.manual_seed(m + dh)
    k, n = 384, heads * dh
    res, g, b = torch.randn(m, k, device=DEV), _param(k), _param(k)
    ws, bs = [_param(n, k) for _ in range(3)], [_param(n) for _ in range(3)]
    slots = torch.randperm(160, device=DEV)[:m].to(torch.int32)
    if m > 2:
        slots[1] = -1               # written nowhere
    kc = torch.zeros(10, heads, 16, dh, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros(10, heads, *((dh, 16) if vt else (16, dh)), device=DEV,
                     dtype=torch.bfloat16)
    want = e.normed_affine(res, g, b, 1e-5, ws, bs)
    got = e.normed_affine(res, g, b, 1e-5, ws, bs, k_cache=kc, v_cache=vc,
                          slots=slots)
    assert len(got) == 1 and torch.equal(got[0], want[0])
    kr, vr = torch.zeros_like(kc), torch.zeros(kc.shape, device=DEV,
                                               dtype=torch.bfloat16)
    for i, t in enumerate(slots.tolist()):
        if t >= 0:
            kr[t // 16, :, t % 16] = want[1][i].view(heads, dh)
            vr[t // 16, :, t % 16] = want[2][i].view(heads, dh)
    assert torch.equal(kc, kr)
    assert torch.equal(vc.transpose(-1, -2) if vt else vc, vr)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(32, 32), (96, 1056), (768, 3072),
                                 (768, 768), (64, 4096)])
def test_added_products(m, n, k):
    """Into an fp32 residual: sums of up to 4096 terms in another order."""
    e = ops.ext()
    torch.manual_seed(m + n)
    x = (torch.randn(m, k, device=DEV) / k ** 0.5).bfloat16()
    w, b = _param(n, k), _param(n)
    res = torch.randn(m, n, device=DEV)
    ref = res.double() + x.double() @ w.double().t() + b.double()
    forms = [e.decode_swizzle_x(x)] + ([x] if e.affine_in_rows(m) else [])
    for form in forms:
        r = res.clone()
        e.affine_add_(form, w, b, r)
        assert _rel(r, ref) < 1e-5


def test_embeddings():
    torch.manual_seed(0)
    table, places = _param(50, 776), _param(20, 776)
    tokens = torch.tensor([0, 49, 7], device=DEV)
    positions = torch.tensor([19, 0, 3], device=DEV, dtype=torch.int32)
    got = ops.ext().embed_res32(tokens, positions, table, places)
    assert torch.equal(got, table[tokens].float() +
                       places[positions.long()].float())


@pytest.mark.parametrize("batch", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("act,bias", [("relu", True), ("gelu_tanh", False)])
def test_decode_step(monkeypatch, batch, act, bias):
    """A step on these kernels and on those with a launch for each norm: some
    ten roundings of 2^-9 a layer, two layers."""
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer, fuse_for_inference
    cfg = ModelConfig("chain", 300, 768, 2, 12, 12, 1536, max_seq_len=80,
                      head_dim=64, norm="layernorm", act=act, pos="learned",
                      attn_bias=bias, mlp_bias=bias)
    torch.manual_seed(batch)
    m = fuse_for_inference(Transformer(cfg, dtype=torch.bfloat16, tp=1)
                           .to(DEV).eval())
    i32 = dict(dtype=torch.int32, device=DEV)
    lens = torch.arange(batch, **i32) * 7 % 70 + 1
    fills = [[torch.randn(batch * 80, 12, 64, device=DEV).bfloat16()
              for _ in "kv"] for _ in m.blocks]

    def step():
        caches = m.alloc_caches(batch * 5, DEV)
        for (kc, vc), (k, v) in zip(caches, fills):
            ops.kv_append(k, v, kc, vc, torch.arange(batch * 80, **i32))
        logits = m.decode(torch.arange(batch, device=DEV), lens - 1, caches,
                          torch.arange(batch, **i32) * 80 + lens - 1,
                          torch.arange(batch * 5, **i32).view(batch, 5), lens)
        return [logits] + [c for layer in caches for c in layer]

    with torch.no_grad():
        calls = []
        chain = m._decode_affine_chain
        monkeypatch.setattr(m, "_decode_affine_chain",
                            lambda *a: calls.append(1) or chain(*a))
        got = step()
        assert calls == [1]
        monkeypatch.setattr(m, "_affine_chain_ready", lambda *a: False)
        for a, b in zip(got, step()):
            assert _rel(a, b.double()) < 2e-2
