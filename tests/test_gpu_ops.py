"""GPU kernel numerics: every gfx950 HIP kernel vs its plain-PyTorch fp32
CPU reference. Run on an MI355X box with `pytest -m gpu`."""
import math
import zlib

import pytest
import torch

from runbooks_amd import ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _assert_hip():
    assert ops.has_hip(), "gfx950 extension must be loaded on the GPU box"


@pytest.mark.parametrize("shape", [(4, 256), (33, 4096), (257, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rmsnorm_fwd(shape, dtype):
    _assert_hip()
    torch.manual_seed(0)
    x = torch.randn(shape, dtype=dtype, device=DEV)
    w = torch.randn(shape[-1], dtype=dtype, device=DEV)
    y = ops.rmsnorm(x, w, 1e-5)
    ref = ops.rmsnorm_ref(x.cpu().float(), w.cpu().float(), 1e-5)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    assert torch.allclose(y.cpu().float(), ref, atol=tol, rtol=tol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rmsnorm_bwd(dtype):
    _assert_hip()
    torch.manual_seed(0)
    N, D = 64, 1024
    xg = torch.randn(N, D, dtype=dtype, device=DEV, requires_grad=True)
    wg = torch.randn(D, dtype=dtype, device=DEV, requires_grad=True)
    dy = torch.randn(N, D, dtype=dtype, device=DEV)
    ops.rmsnorm(xg, wg, 1e-5).backward(dy)

    xc = xg.detach().cpu().float().requires_grad_(True)
    wc = wg.detach().cpu().float().requires_grad_(True)
    ops.rmsnorm_ref(xc, wc, 1e-5).backward(dy.cpu().float())
    tol = 5e-2 if dtype == torch.bfloat16 else 1e-4
    assert torch.allclose(xg.grad.cpu().float(), xc.grad, atol=tol, rtol=tol)
    assert torch.allclose(wg.grad.cpu().float(), wc.grad, atol=tol * 4, rtol=tol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rope_fwd_bwd(dtype):
    _assert_hip()
    torch.manual_seed(0)
    T, H, D = 37, 8, 128
    x = torch.randn(T, H, D, dtype=dtype, device=DEV, requires_grad=True)
    cos, sin = ops.rope_tables(D, 64, device=DEV)
    pos = torch.randint(0, 64, (T,), dtype=torch.int32, device=DEV)
    y = ops.rope(x, cos, sin, pos)
    ref = ops.rope_ref(x.detach().cpu().float(), cos.cpu(), sin.cpu(), pos.cpu())
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    assert torch.allclose(y.detach().cpu().float(), ref, atol=tol, rtol=tol)
    # backward = inverse rotation: rope_bwd(rope_fwd(x)) grads -> dy rotated back
    dy = torch.randn_like(x)
    y.backward(dy)
    ref_grad = ops.rope_ref(dy.cpu().float(), cos.cpu(), -sin.cpu(), pos.cpu())
    assert torch.allclose(x.grad.cpu().float(), ref_grad, atol=tol, rtol=tol)


@pytest.mark.parametrize("pdtype", [torch.float32, torch.bfloat16])
def test_fused_adamw_optimizer(pdtype):
    _assert_hip()
    torch.manual_seed(0)
    n = 4097
    p_gpu = torch.nn.Parameter(torch.randn(n, dtype=pdtype, device=DEV))
    p_cpu = torch.nn.Parameter(p_gpu.detach().cpu().clone())
    o_gpu = ops.FusedAdamW([p_gpu], lr=1e-2, weight_decay=0.1)
    o_cpu = ops.FusedAdamW([p_cpu], lr=1e-2, weight_decay=0.1)
    for i in range(4):
        g = torch.randn(n, dtype=pdtype)
        p_gpu.grad = g.to(DEV)
        p_cpu.grad = g.clone()
        o_gpu.step()
        o_cpu.step()
    tol = 3e-2 if pdtype == torch.bfloat16 else 1e-5
    assert torch.allclose(p_gpu.detach().cpu().float(), p_cpu.detach().float(),
                          atol=tol, rtol=tol)


def test_fused_adamw_multi_tensor_many_params():
    """The one-launch multi-tensor path (adamw_step_multi) over many
    odd-sized params vs the CPU reference optimizer."""
    _assert_hip()
    torch.manual_seed(1)
    sizes = [7, 4096, 16 * 4096, 65536 + 3, 11008]
    ps_gpu = [torch.nn.Parameter(torch.randn(n, dtype=torch.bfloat16,
                                             device=DEV)) for n in sizes]
    ps_cpu = [torch.nn.Parameter(p.detach().cpu().clone()) for p in ps_gpu]
    o_gpu = ops.FusedAdamW(ps_gpu, lr=3e-3, weight_decay=0.05)
    o_cpu = ops.FusedAdamW(ps_cpu, lr=3e-3, weight_decay=0.05)
    # stable grad storage across steps (like DDP bucket views) so the
    # cached chunk table is reused after step 1
    gs = [torch.randn(n, dtype=torch.bfloat16, device=DEV) for n in sizes]
    for pg, g in zip(ps_gpu, gs):
        pg.grad = g
    for _ in range(3):
        for g in gs:
            g.normal_()
        for pc, g in zip(ps_cpu, gs):
            pc.grad = g.cpu().clone()
        o_gpu.step()
        o_cpu.step()
    for pg, pc in zip(ps_gpu, ps_cpu):
        assert torch.allclose(pg.detach().cpu().float(), pc.detach().float(),
                              atol=3e-2, rtol=3e-2)


def test_fused_adamw_kernel_mixed_dtypes():
    """fp32 master params + bf16 grads straight through the kernel."""
    _assert_hip()
    torch.manual_seed(0)
    n = 2049
    p = torch.randn(n, dtype=torch.float32, device=DEV)
    g = torch.randn(n, dtype=torch.bfloat16, device=DEV)
    m = torch.zeros(n, dtype=torch.float32, device=DEV)
    v = torch.zeros(n, dtype=torch.float32, device=DEV)
    p_ref, m_ref, v_ref = p.cpu().clone(), m.cpu().clone(), v.cpu().clone()
    for step in (1, 2):
        ops.ext().adamw_step(p, g, m, v, 1e-2, 0.9, 0.999, 1e-8, 0.1, step)
        # CPU reference math
        gf = g.cpu().float()
        m_ref.mul_(0.9).add_(gf, alpha=0.1)
        v_ref.mul_(0.999).addcmul_(gf, gf, value=0.001)
        bc1, bc2 = 1 - 0.9 ** step, 1 - 0.999 ** step
        p_ref -= 1e-2 * ((m_ref / bc1) / ((v_ref / bc2).sqrt() + 1e-8) + 0.1 * p_ref)
    assert torch.allclose(p.cpu(), p_ref, atol=1e-5, rtol=1e-5)


def test_sample_greedy_matches_argmax():
    _assert_hip()
    torch.manual_seed(0)
    logits = torch.randn(33, 50272, dtype=torch.bfloat16, device=DEV)
    out = ops.sample_tokens(logits, temperature=0.0)
    ref = logits.float().argmax(-1)
    assert torch.equal(out.long().cpu(), ref.cpu())


def test_sample_temperature_distribution():
    _assert_hip()
    # three logits, temperature 1: empirical distribution ~ softmax
    logits = torch.tensor([[2.0, 1.0, 0.0]], device=DEV).repeat(3000, 1)
    out = ops.sample_tokens(logits, temperature=1.0, seed=7).cpu()
    freq = torch.bincount(out.long(), minlength=3).float() / out.numel()
    expect = torch.softmax(torch.tensor([2.0, 1.0, 0.0]), 0)
    assert (freq - expect).abs().max() < 0.05, (freq, expect)


def test_kv_append():
    _assert_hip()
    torch.manual_seed(0)
    Hkv, BS, D, T = 4, 16, 128, 93
    kc = torch.zeros(16, Hkv, BS, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    slots = torch.randperm(16 * BS, device=DEV)[:T].to(torch.int32)
    ops.kv_append(k, v, kc, vc, slots)
    kc_ref = torch.zeros(16, Hkv, BS, D, dtype=torch.bfloat16)
    vc_ref = torch.zeros_like(kc_ref)
    ops.kv_append_ref(k.cpu(), v.cpu(), kc_ref, vc_ref, slots.cpu())
    assert torch.equal(kc.cpu(), kc_ref)
    assert torch.equal(vc.cpu(), vc_ref)


@pytest.mark.parametrize("hq,hkv,dh", [(8, 8, 128), (8, 2, 128), (16, 1, 64),
                                       (64, 8, 128), (4, 4, 64)])
@pytest.mark.parametrize("nsplit", [1, 4])
@pytest.mark.parametrize("vt", [False, True])
def test_paged_decode(hq, hkv, dh, nsplit, vt):
    # vt=True: transposed-V cache layout -> the MFMA decode kernel
    # (only valid for its eligibility set G>=4 / dh<=128)
    if vt and (hq // hkv < 4 or dh > 128):
        pytest.skip("vt layout is MFMA-only (G>=4, dh<=128)")
    _assert_hip()
    torch.manual_seed(hq * 100 + hkv)
    B, BS = 3, 16
    seq_lens = torch.tensor([5, 333, 170], dtype=torch.int32)
    n_blocks = int(sum((int(s) + BS - 1) // BS for s in seq_lens)) + 2
    kc = torch.randn(n_blocks, hkv, BS, dh, dtype=torch.bfloat16, device=DEV)
    vc = torch.randn_like(kc)
    maxb = (int(seq_lens.max()) + BS - 1) // BS
    bt = torch.zeros(B, maxb, dtype=torch.int32)
    nxt = 0
    for b in range(B):
        nb = (int(seq_lens[b]) + BS - 1) // BS
        bt[b, :nb] = torch.arange(nxt, nxt + nb, dtype=torch.int32)
        nxt += nb
    q = torch.randn(B, hq, dh, dtype=torch.bfloat16, device=DEV)
    scale = 1 / math.sqrt(dh)
    vc_dev = vc.permute(0, 1, 3, 2).contiguous() if vt else vc
    out = ops.paged_decode(q, kc, vc_dev, bt.to(DEV), seq_lens.to(DEV),
                           scale=scale, nsplit=nsplit)
    ref = ops.paged_decode_ref(q.cpu().float(), kc.cpu().float(), vc.cpu().float(),
                               bt, seq_lens, scale)
    assert torch.allclose(out.cpu().float(), ref, atol=3e-2, rtol=3e-2), \
        (out.cpu().float() - ref).abs().max()


@pytest.mark.parametrize("fused", [False, True])
def test_kv_append_v_transposed(fused):
    """kv_append / qkv_rope_append into the transposed-V layout match the
    plain layout element-for-element."""
    _assert_hip()
    torch.manual_seed(3)
    hkv, dh, BS, nb = 8, 128, 16, 6
    T = 21
    k = torch.randn(T, hkv, dh, dtype=torch.bfloat16, device=DEV)
    v = torch.randn(T, hkv, dh, dtype=torch.bfloat16, device=DEV)
    slots = torch.arange(3, 3 + T, dtype=torch.int32, device=DEV)
    kc1, vc1 = ops.alloc_kv_cache(nb, hkv, dh, DEV)
    kc2, vc2 = ops.alloc_kv_cache(nb, hkv, dh, DEV, v_transposed=True)
    if fused:
        hq = 16
        y = torch.randn(T, (hq + 2 * hkv) * dh, dtype=torch.bfloat16,
                        device=DEV)
        pos = torch.arange(T, dtype=torch.int32, device=DEV)
        from runbooks_amd.ops.rope import rope_tables
        cos, sin = rope_tables(dh, 64, 10000.0, DEV)
        q1 = ops.ext().qkv_rope_append(y, cos, sin, pos, kc1, vc1, slots, hq)
        q2 = ops.ext().qkv_rope_append(y, cos, sin, pos, kc2, vc2, slots, hq)
        assert torch.equal(q1, q2)
    else:
        ops.kv_append(k, v, kc1, vc1, slots)
        ops.kv_append(k, v, kc2, vc2, slots)
    assert torch.equal(kc1, kc2)
    assert torch.equal(vc1, vc2.permute(0, 1, 3, 2).contiguous())


def test_engine_gpu_matches_full_forward():
    """Greedy decode through the paged HIP kernels == full no-cache forward."""
    _assert_hip()
    from runbooks_amd.models import build_model
    from runbooks_amd.serve import Engine

    m = build_model("smoke-llama", dtype=torch.bfloat16, device=DEV)
    eng = Engine(m, device=DEV, kv_blocks=128)
    prompt = [5, 9, 2, 7, 1, 3]
    out = eng.generate(list(prompt), max_new_tokens=6)
    seq = list(prompt)
    for _ in range(6):
        logits = m(torch.tensor([seq], device=DEV))
        seq.append(int(logits[0, -1].argmax()))
    assert out == seq[len(prompt):], (out, seq[len(prompt):])


def test_train_step_gpu():
    from runbooks_amd.train import TrainConfig, Trainer

    cfg = TrainConfig(model="smoke-llama", seq_len=64, micro_batch=2,
                      num_train_steps=8, dtype="bfloat16", lr=1e-3)
    tr = Trainer(cfg, device=DEV)
    torch.manual_seed(0)
    batch = torch.randint(0, 512, (2, 65))
    losses = [tr.train_step(batch) for _ in range(8)]
    assert losses[-1] < losses[0], losses
    assert all(math.isfinite(x) for x in losses)


@pytest.mark.parametrize("M,N,K", [
    (1, 4096, 4096),       # batch-1 decode qkv/o
    (32, 4096, 4096),      # full bucket
    (32, 11008, 4096),     # mlp up
    (32, 4096, 11008),     # mlp down (odd K split)
    (17, 32000, 4096),     # lm_head, ragged M
    (8, 128, 256),         # minimal grid
    (32, 4096, 512),       # falcon-7b-ish head shard
])
def test_skinny_gemm(M, N, K):
    """csrc/skinny_gemm.hip vs fp32 matmul."""
    _assert_hip()
    torch.manual_seed(M * 31 + N)
    x = torch.randn(M, K, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(N, K, dtype=torch.bfloat16, device=DEV)
    y = ops.ext().skinny_gemm(x, w)
    ref = x.cpu().float() @ w.cpu().float().t()
    d = (y.cpu().float() - ref).abs().max().item()
    rel = d / ref.abs().max().item()
    assert rel < 2e-2, f"max abs {d} rel {rel}"


def test_fast_linear_dispatch():
    """fast_linear uses the skinny kernel only on decode shapes."""
    _assert_hip()
    x = torch.randn(4, 256, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(128, 256, dtype=torch.bfloat16, device=DEV)
    with torch.no_grad():
        y = ops.fast_linear(x, w)
    ref = (x.float() @ w.float().t())
    assert (y.float() - ref).abs().max() < ref.abs().max() * 2e-2
    # grad-enabled path must stay on the library (autograd-able)
    xg = x.clone().requires_grad_(True)
    y2 = ops.fast_linear(xg, w)
    y2.sum().backward()
    assert xg.grad is not None


@pytest.mark.parametrize("hq,hkv,dh", [(8, 8, 128), (8, 2, 128), (16, 1, 64)])
def test_qkv_rope_append(hq, hkv, dh):
    """Fused packed-qkv epilogue vs the composed rope + kv_append ops."""
    _assert_hip()
    torch.manual_seed(hq)
    T, BS, nblocks = 7, 16, 8
    y = torch.randn(T, (hq + 2 * hkv) * dh, dtype=torch.bfloat16, device=DEV)
    cos, sin = ops.rope_tables(dh, 64, device=DEV)
    pos = torch.randint(0, 64, (T,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(nblocks * BS, device=DEV)[:T].to(torch.int32)

    kc = torch.zeros(nblocks, hkv, BS, dh, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    q = ops.ext().qkv_rope_append(y, cos, sin, pos, kc, vc, slots, hq)

    qo, kvo = hq * dh, hkv * dh
    q_ref = ops.rope(y[:, :qo].contiguous().view(T, hq, dh), cos, sin, pos)
    k_ref = ops.rope(y[:, qo:qo + kvo].contiguous().view(T, hkv, dh),
                     cos, sin, pos)
    v_ref = y[:, qo + kvo:].contiguous().view(T, hkv, dh)
    kc_ref = torch.zeros_like(kc)
    vc_ref = torch.zeros_like(vc)
    ops.kv_append(k_ref, v_ref, kc_ref, vc_ref, slots)

    assert torch.allclose(q.float(), q_ref.float(), atol=2e-2, rtol=2e-2)
    assert torch.allclose(kc.float(), kc_ref.float(), atol=2e-2, rtol=2e-2)
    assert torch.equal(vc, vc_ref)


def test_swiglu_packed():
    _assert_hip()
    torch.manual_seed(0)
    y = torch.randn(33, 2 * 1024, dtype=torch.bfloat16, device=DEV)
    out = ops.ext().swiglu_packed(y)
    g, u = y[:, :1024].contiguous(), y[:, 1024:].contiguous()
    ref = torch.nn.functional.silu(g.float()) * u.float()
    assert torch.allclose(out.float(), ref, atol=2e-2, rtol=2e-2)


def test_mfma_32x32x16_layout_probe():
    """One MFMA vs torch matmul — pinpoints a wrong fragment map."""
    _assert_hip()
    torch.manual_seed(0)
    # asymmetric inputs (guide: symmetric B passes transposed layouts)
    a = torch.randn(32, 16, dtype=torch.bfloat16, device=DEV)
    b = torch.arange(16 * 32, dtype=torch.float32, device=DEV).reshape(16, 32)
    b = ((b % 13) / 6.0 - 1.0).to(torch.bfloat16)
    c = ops.ext().mfma_probe_32x32x16(a, b)
    ref = a.float() @ b.float()
    assert torch.allclose(c, ref, atol=2e-2, rtol=2e-2), \
        (c - ref).abs().max()


@pytest.mark.parametrize("B,S,Hq,Hkv,dh", [
    (1, 64, 4, 4, 128),      # tiny, single WG tile
    (2, 333, 8, 2, 128),     # ragged S, GQA
    (1, 511, 16, 1, 64),     # MQA falcon-style, Dh=64
    (2, 1024, 8, 8, 128),    # multi-tile
])
def test_flash_prefill(B, S, Hq, Hkv, dh):
    _assert_hip()
    torch.manual_seed(B * 1000 + S)
    q = torch.randn(B, S, Hq, dh, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(B, S, Hkv, dh, dtype=torch.bfloat16, device=DEV)
    v = torch.randn(B, S, Hkv, dh, dtype=torch.bfloat16, device=DEV)
    out = ops.flash_prefill(q, k, v)
    ref = ops.causal_attention(q.cpu().float(), k.cpu().float(), v.cpu().float())
    diff = (out.cpu().float() - ref).abs().max()
    assert diff < 3e-2, f"max diff {diff}"


@pytest.mark.parametrize("B,S,Hq,Hkv,dh,scale", [
    # up to 512 tiles of 32 rows, two waves a tile
    (1, 1, 2, 1, 64, None), (2, 33, 3, 3, 128, -0.1), (1, 65, 2, 1, 128, 0.0),
    # up to 1536 tiles, four waves
    (1, 545, 32, 8, 64, None), (2, 257, 40, 8, 128, None),
    (1, 63, 4, 2, 256, None), (1, 321, 24, 8, 256, -0.05),
    # one wave a tile
    (1, 1601, 32, 8, 128, None), (2, 737, 32, 32, 64, None),
    (1, 1313, 32, 32, 256, None),
    # eight waves
    (1, 1537, 128, 8, 64, None), (3, 1025, 64, 2, 128, None),
    (1, 6209, 32, 8, 128, None), (6, 320, 128, 64, 64, None),
    (6, 288, 128, 64, 128, 0.0)])
def test_flash_prefill_tiles(B, S, Hq, Hkv, dh, scale):
    """Every split of the rows over waves, at remainders of its tiles, with
    inputs that start off a 16-byte boundary. Weights and result are rounded to
    bf16 (2^-9 relative each), sums are fp32."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(S)

    def rows(h):
        n = B * S * h * dh
        return torch.randn(n + 1, generator=g, device=DEV).bfloat16()[1:] \
            .view(B, S, h, dh)

    q, k, v = rows(Hq), rows(Hkv), rows(Hkv)
    scale = dh ** -0.5 if scale is None else scale
    out, lse = ops.ext().flash_fwd_train(q, k, v, scale)
    hidden = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1)
    for h in {0, Hq // 2, Hq - 1}:
        at = h // (Hq // Hkv)
        for b in range(B):
            s = q[b, :, h].double() @ k[b, :, at].double().t() * scale
            s = s.masked_fill(hidden, float("-inf"))
            ref = s.softmax(-1) @ v[b, :, at].double()
            assert (out[b, :, h] - ref).norm() < 2 ** -8 * ref.norm()
            assert (lse[b, h] - s.logsumexp(-1)).abs().max() < 1e-5


def _hashed(n, salt):
    """Values in [-2, 2) that are the same everywhere."""
    i = torch.arange(n, dtype=torch.int64) + salt * 7919
    h = (i * 2654435761) & 0xffffffff
    h = ((h >> 15) ^ h) * 2246822519 & 0xffffffff
    h = (h >> 13) ^ h
    return ((h & 0xffff).float() / 65536 - 0.5) * 4


@pytest.mark.parametrize("S,hq,dh", [(160, 4, 64), (160, 4, 128), (97, 4, 256),
                                     (330, 4, 256), (1313, 32, 256)])
def test_flash_rising_scores(S, hq, dh):
    """Scores that rise with the key, so that every tile moves the maximum and with it
    the sums before it, to nearly nothing: rounded probabilities and results."""
    _assert_hip()
    torch.manual_seed(dh)
    q = torch.full((1, S, hq, dh), 0.5, device=DEV).bfloat16()
    k = (torch.arange(S, device=DEV) / (8 * dh ** 0.5))[None, :, None, None] \
        .expand(1, S, hq, dh).bfloat16().contiguous()
    v = torch.randn(1, S, hq, dh, device=DEV).bfloat16()
    out = ops.ext().flash_prefill(q, k, v, 4.0)
    for h in range(0, hq, 7):
        s = q[0, :, h].double() @ k[0, :, h].double().t() * 4.0
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1),
                          -torch.inf)
        ref = s.softmax(-1) @ v[0, :, h].double()
        assert (out[0, :, h].double() - ref).norm() <= 2 ** -7 * ref.norm()


@pytest.mark.parametrize("dh", [64, 128, 256])
@pytest.mark.parametrize("S,hq", [(33, 1), (160, 4), (330, 4), (1313, 32)])
def test_flash_rows_beside_one_that_jumps(S, hq, dh):
    """One row of every 32 whose scores rise by 12 exponents of 2 with each 32 keys,
    which moves the maxima of all of them, while the others rise by 0.5 to 3: their sums
    so far are scaled by 0.125 to 0.7 each time, and stay part of the result."""
    _assert_hip()
    torch.manual_seed(dh)
    steps = torch.arange(S, device=DEV) // 32
    rise = (0.5 + 2.5 * torch.rand(int(steps[-1]) + 1, device=DEV)).cumsum(0)
    q = 0.3 * torch.randn(1, S, hq, dh, device=DEV)
    k = 0.3 * torch.randn(1, S, hq, dh, device=DEV)
    jumps = torch.arange(S, device=DEV) % 32 == 9
    q[..., 0], q[..., 1] = (~jumps)[None, :, None], jumps[None, :, None]
    unit = math.log(2) * dh ** 0.5
    k[..., 0] = (rise[steps] * unit)[None, :, None]
    k[..., 1] = (12 * steps * unit)[None, :, None]
    q, k = q.bfloat16(), k.bfloat16()
    v = torch.randn(1, S, hq, dh, device=DEV).bfloat16()
    out = ops.ext().flash_prefill(q, k, v, dh ** -0.5)
    for h in range(0, hq, 7):
        s = q[0, :, h].double() @ k[0, :, h].double().t() * dh ** -0.5
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1),
                          -torch.inf)
        ref = s.softmax(-1) @ v[0, :, h].double()
        off = (out[0, :, h].double() - ref).norm(dim=-1)
        assert bool((off <= 2 ** -6 * ref.norm(dim=-1)).all())


@pytest.mark.parametrize("B,S,Hq,Hkv,bits", [
    (1, 1, 1, 1, (4093165637, 932004135, 3265854109, 3265854109, 34914089)),
    (2, 31, 3, 3, (2980831709, 3346004597, 2951792153, 627292471,
                   1842450457)),
    (1, 64, 4, 2, (3987702248, 4086934317, 3359148874, 2069512852,
                   558976727)),
    (1, 65, 12, 12, (329763779, 1455785953, 2509830808, 4046418718,
                     123667421)),
    (2, 257, 12, 12, (1483102084, 2568763203, 2368670429, 1348113486,
                      3775892656)),
    (1, 300, 4, 1, (2206580616, 3272915928, 1571533394, 3616146700,
                    1162676308)),
    (1, 1021, 12, 12, (277277627, 2214567642, 3491892497, 2225167499,
                       4002099437))])
def test_flash_ordered_bits(B, S, Hq, Hkv, bits):
    """The attention that ReLU models train on does not change a bit of its
    result, log-sum-exp and gradients (their CRCs), as the model's gradients
    and the weights of later steps would follow."""
    _assert_hip()
    q, k, v, dout = (_hashed(B * S * h * 64, salt).view(B, S, h, 64)
                     .bfloat16().to(DEV).requires_grad_()
                     for salt, h in ((1, Hq), (2, Hkv), (3, Hkv), (4, Hq)))
    out, lse = ops.ext().flash_fwd_train(q, k, v, 0.125, ordered=True)
    grads = ops.ext().fa_bwd(dout, q, k, v, out, lse, 0.125, ordered=True)
    crc = [zlib.crc32(x.detach().cpu().numpy().tobytes()) for x in
           (out.view(torch.int16), lse, *(g.view(torch.int16)
                                          for g in grads))]
    assert tuple(crc) == bits
    y = ops.causal_attention(q, k, v, ordered=True)
    y.backward(dout.detach())
    assert torch.equal(y, out) and torch.equal(q.grad, grads[0])


@pytest.mark.parametrize("S,scale", [(97, None), (200, -0.1), (130, 0.0),
                                     (33, 0.3)])
def test_flash_ordered(S, scale):
    """As test_flash_prefill_tiles and test_flash_attention_bwd_tiles, with any
    factor."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(S)
    q, k, v, dout = (torch.randn(2, S, h, 64, generator=g, device=DEV)
                     .bfloat16() for h in (6, 3, 3, 6))
    scale = 0.125 if scale is None else scale
    out, lse = ops.ext().flash_fwd_train(q, k, v, scale, ordered=True)
    ref = q.double().transpose(1, 2) @ k.double().repeat_interleave(
        2, 2).permute(0, 2, 3, 1).contiguous() * scale
    ref.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1),
                     float("-inf"))
    assert (lse - ref.logsumexp(-1)).abs().max() < 1e-5
    p, vs = ref.softmax(-1), v.double().repeat_interleave(2, 2).transpose(
        1, 2).contiguous()
    ref = p @ vs
    assert (out.transpose(1, 2) - ref).norm() < 2 ** -8 * ref.norm()
    got = ops.ext().fa_bwd(dout, q, k, v, out, lse, scale, ordered=True)
    for b in range(2):
        for h in range(6):
            qs, ks, do, o = (x[b, :, i].double() for x, i in (
                (q, h), (k, h // 2), (dout, h), (out, h)))
            w = p[b, h]
            ds = w * (do @ vs[b, h].t() -
                      (do * o).sum(-1, keepdim=True)) * scale
            for x, r in zip(got, (ds @ ks, ds.t() @ qs, w.t() @ do)):
                assert (x[b, :, h] - r).norm() <= 2 ** -7 * r.norm()


@pytest.mark.parametrize("B,S,Hq,Hkv,dh,scale", [
    # up to 512 tiles of 32 rows, workgroups of 64 rows
    (1, 2, 2, 1, 64, None), (2, 33, 3, 3, 128, -0.1), (1, 65, 2, 1, 128, 0.0),
    (1, 97, 12, 12, 64, None),
    # of 128 rows
    (1, 545, 32, 8, 64, None), (2, 257, 40, 8, 128, None),
    (3, 1001, 8, 8, 128, -0.05)])
def test_flash_attention_bwd_tiles(B, S, Hq, Hkv, dh, scale):
    """Gradients at remainders of the tiles, inputs off a 16-byte boundary,
    from the result that the forward rounded. At most two roundings to bf16
    (2^-9 relative) lie on the way to one; differences of dO V^T and D may be
    half of their terms."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(S)

    def rows(h):
        n = B * S * h * dh
        return torch.randn(n + 1, generator=g, device=DEV).bfloat16()[1:] \
            .view(B, S, h, dh)

    q, k, v, dout = rows(Hq), rows(Hkv), rows(Hkv), rows(Hq)
    scale = dh ** -0.5 if scale is None else scale
    out, lse = ops.ext().flash_fwd_train(q, k, v, scale)
    got = ops.ext().fa_bwd(dout, q, k, v, out, lse, scale)
    hidden = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1)
    for h in {0, Hq // 2, Hq - 1}:
        at = h // (Hq // Hkv)
        for b in range(B):
            qs, ks, vs, do, o = (x[b, :, i].double() for x, i in (
                (q, h), (k, at), (v, at), (dout, h), (out, h)))
            p = (qs @ ks.t() * scale).masked_fill(
                hidden, float("-inf")).softmax(-1)
            ds = p * (do @ vs.t() - (do * o).sum(-1, keepdim=True)) * scale
            for x, ref in zip(got, (ds @ ks, ds.t() @ qs, p.t() @ do)):
                assert (x[b, :, h] - ref).norm() <= 2 ** -7 * ref.norm()


@pytest.mark.parametrize("B,S,Hq,Hkv,dh", [
    (1, 64, 4, 4, 128),      # tiny, single WG tile
    (2, 333, 8, 2, 128),     # ragged S, GQA (group-summed dk/dv)
    (1, 200, 8, 1, 64),      # MQA, Dh=64
    (1, 576, 4, 4, 128),     # multi-WG, MHA (llama2-7b shape class)
])
def test_flash_attention_train_bwd(B, S, Hq, Hkv, dh):
    """fa_bwd (attention_bwd.hip) vs torch autograd through the fp32
    reference attention."""
    _assert_hip()
    torch.manual_seed(B * 77 + S)
    q = torch.randn(B, S, Hq, dh, dtype=torch.bfloat16, device=DEV,
                    requires_grad=True)
    k = torch.randn(B, S, Hkv, dh, dtype=torch.bfloat16, device=DEV,
                    requires_grad=True)
    v = torch.randn(B, S, Hkv, dh, dtype=torch.bfloat16, device=DEV,
                    requires_grad=True)
    out = ops.causal_attention(q, k, v)   # MFMA autograd path on GPU
    dy = torch.randn_like(out)
    out.backward(dy)

    qc = q.detach().cpu().float().requires_grad_(True)
    kc = k.detach().cpu().float().requires_grad_(True)
    vc = v.detach().cpu().float().requires_grad_(True)
    ref = ops.causal_attention(qc, kc, vc)
    ref.backward(dy.cpu().float())

    assert (out.detach().cpu().float() - ref.detach()).abs().max() < 3e-2
    for got, want, name in ((q.grad, qc.grad, "dq"), (k.grad, kc.grad, "dk"),
                            (v.grad, vc.grad, "dv")):
        g = got.cpu().float()
        d = (g - want).abs().max().item()
        rel = d / max(want.abs().max().item(), 1e-6)
        assert rel < 4e-2, f"{name}: max abs diff {d} rel {rel}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_swiglu_fwd_bwd(dtype):
    _assert_hip()
    torch.manual_seed(0)
    g = torch.randn(64, 1024, dtype=dtype, device=DEV, requires_grad=True)
    u = torch.randn(64, 1024, dtype=dtype, device=DEV, requires_grad=True)
    y = ops.swiglu(g, u)
    dy = torch.randn_like(y)
    y.backward(dy)
    gc = g.detach().cpu().float().requires_grad_(True)
    uc = u.detach().cpu().float().requires_grad_(True)
    yc = torch.nn.functional.silu(gc) * uc
    yc.backward(dy.cpu().float())
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    assert torch.allclose(y.detach().cpu().float(), yc.detach(), atol=tol, rtol=tol)
    assert torch.allclose(g.grad.cpu().float(), gc.grad, atol=tol, rtol=tol)
    assert torch.allclose(u.grad.cpu().float(), uc.grad, atol=tol, rtol=tol)


@pytest.mark.parametrize("V", [32000, 50272])
def test_cross_entropy_fwd_bwd(V):
    _assert_hip()
    torch.manual_seed(0)
    N = 37
    logits = torch.randn(N, V, dtype=torch.bfloat16, device=DEV,
                         requires_grad=True)
    targets = torch.randint(0, V, (N,), device=DEV)
    targets[3] = -100  # ignore_index
    loss = ops.cross_entropy(logits, targets)
    loss.backward()
    lc = logits.detach().cpu().float().requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(lc, targets.cpu().long(),
                                            ignore_index=-100)
    ref.backward()
    assert abs(float(loss) - float(ref)) < 2e-2, (float(loss), float(ref))
    assert torch.allclose(logits.grad.cpu().float(), lc.grad, atol=2e-3,
                          rtol=2e-2), (logits.grad.cpu().float() - lc.grad).abs().max()


@pytest.mark.parametrize("M,N,K", [
    (1, 64, 256), (2, 96, 32), (7, 4096, 11008), (16, 12288, 4096),
    (31, 4096, 4096), (32, 22016, 2080)])
def test_decode_gemm_fp8(M, N, K):
    """Both outputs against the product with the dequantized weights: exact
    products, fp32 sums (their order: 1e-5), y rounded to bf16."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w8 = torch.randn(N, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    scale = torch.rand(N, generator=g, device=DEV) + 0.5
    ref = x.double() @ (w8.double() * scale.double()[:, None]).t()
    e = ops.ext()
    args = (e.decode_swizzle_x(x), e.decode_swizzle_w8(w8.view(torch.uint8)),
            scale, M, N, K)
    assert (e.decode_gemm_fp8(*args) - ref).norm() < 2 ** -8 * ref.norm()
    raw = e.decode_gemm_fp8(*args, raw=True)
    split = e.decode_gemm_split(N, K)
    assert raw.dtype == (torch.float32 if split > 1 else torch.bfloat16)
    if split > 1:
        assert (raw.double().sum(0) - ref).norm() < 1e-5 * ref.norm()


def test_skinny_gemm_fp8():
    """fp8 weight-only decode GEMM vs matmul on the dequantized weights
    (exact dequant path) and vs the original bf16 weights (e4m3 bound)."""
    _assert_hip()
    from runbooks_amd.ops.linear import dequantize_fp8, quantize_fp8, _FP8_REGISTRY
    torch.manual_seed(4)
    M, N, K = 32, 4096, 4096
    x = torch.randn(M, K, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(N, K, dtype=torch.bfloat16, device=DEV)
    w8, scale = quantize_fp8(w)
    y = ops.ext().skinny_gemm_fp8(x, w8, scale)
    deq = dequantize_fp8(w8, scale).to(DEV)
    ref = (x.float() @ deq.float().t())
    d = (y.float() - ref).abs().max() / ref.abs().max()
    assert d < 2e-2, f"vs dequant rel {d}"
    full = (x.float() @ w.float().t())
    d2 = (y.float() - full).abs().max() / full.abs().max()
    assert d2 < 0.08, f"vs bf16 rel {d2}"
    _FP8_REGISTRY.clear()


@pytest.mark.parametrize("m", [1, 16, 32])
def test_fp8_weights_as_served(m):
    """The e4m3 weights that models run on, through the dispatch: one rounding
    of the product with the dequantized ones."""
    _assert_hip()
    from runbooks_amd.ops.linear import (decode_linear_raw, dequantize_fp8,
                                         quantize_fp8)
    torch.manual_seed(m)
    x = torch.randn(m, 1024, device=DEV).bfloat16()
    w = torch.randn(4096, 1024, device=DEV).bfloat16()
    deq = dequantize_fp8(*quantize_fp8(w), dtype=torch.float32)
    ref = x.double() @ deq.double().t()
    with torch.no_grad():
        raw = decode_linear_raw(x, w)[0].double()
        for y in (ops.fast_linear(x, w), raw.sum(0) if raw.dim() == 3
                  else raw):
            assert (y - ref).norm() < 2 ** -8 * ref.norm()


_EXPERIMENTAL = __import__("os").environ.get("RB_EXPERIMENTAL") == "1"


def test_mfma_16x16x32_layout_probe():
    _assert_hip()
    torch.manual_seed(0)
    a = torch.randn(16, 32, dtype=torch.bfloat16, device=DEV)
    b = torch.arange(32 * 16, dtype=torch.float32, device=DEV).reshape(32, 16)
    b = ((b % 11) / 5.0 - 1.0).to(torch.bfloat16)   # asymmetric
    c = ops.ext().mfma_probe_16x16x32(a, b)
    ref = a.float() @ b.float()
    assert torch.allclose(c, ref, atol=2e-2, rtol=2e-2), (c - ref).abs().max()


@pytest.mark.skipif(not _EXPERIMENTAL, reason="RB_EXPERIMENTAL=1 only")
@pytest.mark.parametrize("M,N,K", [
    (256, 256, 128),      # single tile, 2 K-tiles (minimum)
    (256, 256, 512),
    (512, 768, 1024),     # multi-tile, XCD remap with nwg%8 != 0
    (512, 768, 4096),     # bisect: deep K alone
    (2048, 4096, 1024),   # bisect: big M*N alone
    (256, 256, 4096),     # bisect: single tile, deep K
    (2048, 4096, 4096),   # the training shape (failed r1: rel 1.29)
])
def test_train_gemm_nt(M, N, K):
    _assert_hip()
    torch.manual_seed(M + N)
    a = torch.randn(M, K, dtype=torch.bfloat16, device=DEV)
    b = torch.randn(N, K, dtype=torch.bfloat16, device=DEV)
    c = ops.ext().train_gemm_nt(a, b)
    ref = (a.float() @ b.float().t())
    d = (c.float() - ref).abs().max().item()
    rel = d / ref.abs().max().item()
    assert rel < 2e-2, f"max abs {d} rel {rel}"


@pytest.mark.gpu
@pytest.mark.skipif(not _EXPERIMENTAL, reason="RB_EXPERIMENTAL=1 only "
                    "(geglu_packed awaits its first on-GPU validation)")
def test_geglu_packed():
    """csrc geglu_packed vs fp32 tanh-gelu reference."""
    from runbooks_amd import ops
    torch.manual_seed(0)
    y = torch.randn(64, 2 * 256, device="cuda", dtype=torch.bfloat16)
    got = ops.ext().geglu_packed(y)
    g, u = y[:, :256].float(), y[:, 256:].float()
    ref = torch.nn.functional.gelu(g, approximate="tanh") * u
    assert torch.allclose(got.float(), ref, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T,hq,hkv,dh,vt", [
    (1, 4, 4, 128, False), (33, 2, 1, 256, False), (63, 8, 2, 64, True),
    (64, 8, 2, 128, True), (65, 4, 1, 64, True), (200, 16, 4, 128, True)])
def test_qkv_rope_append_layouts(T, hq, hkv, dh, vt, fp8):
    """Rotation in place and to a tensor, into every cache layout; tokens that
    fill cache blocks in order, out of order and not at all."""
    _assert_hip()
    from runbooks_amd.ops.kvcache import alloc_kv_cache, fp8_dequant_cache_ref
    g = torch.Generator().manual_seed(T + dh)
    y = torch.randn(T, (hq + 2 * hkv) * dh, generator=g).bfloat16()
    cos, sin = ops.rope_tables(dh, 512)
    pos = torch.randint(0, 512, (T,), generator=g, dtype=torch.int32)
    n = T // 16 + 3
    slots = torch.cat([16 * b + torch.arange(16) for b in
                       torch.randperm(n, generator=g).tolist()])[:T].int()
    if T > 40:
        slots[17:30] = slots[17:30].flip(0)
    if T > 1:
        slots[T // 2] = -1
    q, k, v = (x.view(T, -1, dh) for x in
               y.split([hq * dh, hkv * dh, hkv * dh], -1))
    q, k = (ops.rope_ref(x, cos, sin, pos) for x in (q, k))
    kc, vc = alloc_kv_cache(n, hkv, dh, "cpu", fp8=fp8, v_transposed=vt)
    got = [c.to(DEV) for c in (kc, vc)]
    ops.kv_append_ref(k, v, kc, vc, slots)
    args = (cos.to(DEV), sin.to(DEV), pos.to(DEV), *got, slots.to(DEV), hq)
    qd = ops.ext().qkv_rope_append(y.to(DEV), *args)
    # one rounding apart where the fused multiply-adds differ
    assert (qd.cpu().float() - q.float()).abs().max() <= 2 ** -6

    def check():
        for c, ref in zip(got, (kc, vc)):
            if fp8:
                a, b = (fp8_dequant_cache_ref(x) for x in (c.cpu(), ref))
                # a rounding to e4m3 (2^-3 of the value) may fall otherwise
                assert ((a - b).abs() <= b.abs() / 8 + 1e-2).all()
                assert (a - b).norm() <= 0.01 * b.norm()
            else:
                assert (c.cpu().float() - ref.float()).abs().max() <= 2 ** -6

    check()
    for c in got:
        c.zero_()
    yd = y.to(DEV)
    ops.ext().qkv_rope_append_(yd, *args)
    check()
    want = torch.cat([x.reshape(T, -1) for x in (q, k, v)], -1)
    assert (yd.cpu().float() - want.float()).abs().max() <= 2 ** -6


def test_flash_prefill_qkv():
    """q, k and v read side by side are read as if apart."""
    _assert_hip()
    y = torch.randn(2 * 77, (8 + 2 * 2) * 64, device=DEV).bfloat16()
    q, k, v = (x.reshape(2, 77, -1, 64) for x in y.split([512, 128, 128], -1))
    assert torch.equal(ops.ext().flash_prefill_qkv(y, 2, 77, 8, 2, 64, 0.125),
                       ops.flash_prefill(q, k, v, 0.125))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,D", [
    (1, 8), (3, 2048), (5, 2056), (700, 768), (2, 4544), (33, 8192),
    (2, 8200)])
def test_rmsnorm_residual(rows, D, dtype):
    """Sum and norm forward and backward, a row in 1, 2 and 4 vectors a thread
    and wider; weights with and without gradient."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(D)
    x, d, ds, dy = (torch.randn(rows, D, generator=g, device=DEV).to(dtype)
                    for _ in range(4))
    w = (1 + 0.1 * torch.randn(D, generator=g, device=DEV)).to(dtype)
    tol = 1e-5 if dtype == torch.float32 else 2 ** -7
    ref = [t.double().requires_grad_() for t in (x, d, w)]
    s = ref[0] + ref[1]
    y = s * (s.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * ref[2]
    torch.autograd.backward([s, y], [ds.double(), dy.double()])
    for trains in (True, False):
        leaves = [t.clone().requires_grad_() for t in (x, d)]
        wt = w.clone().requires_grad_(trains)
        got = ops.rmsnorm_res(*leaves, wt, 1e-5)
        torch.autograd.backward(got, [ds, dy])
        pairs = list(zip(got, (s, y))) + list(zip(
            [t.grad for t in leaves], [t.grad for t in ref]))
        if trains:
            pairs.append((wt.grad, ref[2].grad))
        else:
            assert wt.grad is None
        for a, b in pairs:
            assert (a.double() - b).norm() <= tol * b.norm()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,dh,vt", [
    (4, 4, 128, False), (4, 2, 64, False), (2, 2, 256, False),
    (8, 2, 128, True), (16, 1, 64, True), (8, 1, 128, True),
    (8, 2, 128, False)])
def test_paged_decode_steps(hq, hkv, dh, vt, fp8):
    """Lengths around the tokens of a step (8 and 32 of a wave, four waves),
    splits that leave parts empty, starts inside a block."""
    _assert_hip()
    from runbooks_amd.ops.kvcache import alloc_kv_cache
    g = torch.Generator().manual_seed(dh + hq)
    lens = [1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 129, 200]
    B, wide = len(lens), 14
    n = B * wide
    kc, vc = alloc_kv_cache(n, hkv, dh, "cpu", fp8=fp8, v_transposed=vt)
    k, v = (torch.randn(n * 16, hkv, dh, generator=g).bfloat16()
            for _ in range(2))
    ops.kv_append_ref(k, v, kc, vc, torch.arange(n * 16))
    bt = torch.randperm(n, generator=g).view(B, wide).int()
    sl = torch.tensor(lens, dtype=torch.int32)
    starts = torch.tensor([x // 3 for x in lens], dtype=torch.int32)
    q = torch.randn(B, hq, dh, generator=g).bfloat16()
    for st in (None, starts):
        ref = ops.paged_decode_ref(q.float(), kc if fp8 else kc.float(),
                                   vc if fp8 else vc.float(), bt, sl,
                                   dh ** -0.5, seq_starts=st)
        for nsplit in (1, 2, 16):
            got = ops.paged_decode(
                q.to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), sl.to(DEV),
                nsplit=nsplit,
                seq_starts=None if st is None else st.to(DEV))
            # weights (MFMA path) and result rounded to bf16, values up to 5
            assert (got.cpu().float() - ref).abs().max() < 3e-2


@pytest.mark.gpu
@pytest.mark.skipif(not _EXPERIMENTAL, reason="RB_EXPERIMENTAL=1 only "
                    "(Dh=256 decode instantiation awaits GPU validation)")
def test_paged_decode_dh256():
    """gemma-width decode heads: Dh=256 template vs fp32 reference."""
    from runbooks_amd import ops
    torch.manual_seed(0)
    B, hkv, G, bs, nblk, dh = 2, 2, 1, 16, 8, 256
    q = torch.randn(B, hkv * G, dh, device="cuda", dtype=torch.bfloat16)
    kc = torch.randn(nblk, hkv, bs, dh, device="cuda", dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    bt = torch.tensor([[0, 1, 2], [3, 4, 5]], device="cuda",
                      dtype=torch.int32)
    sl = torch.tensor([40, 23], device="cuda", dtype=torch.int32)
    got = ops.paged_decode(q, kc, vc, bt, sl)
    ref = ops.paged_decode_ref(q.float().cpu(), kc.float().cpu(),
                               vc.float().cpu(), bt.cpu(), sl.cpu(),
                               scale=1.0 / 16.0)
    assert torch.allclose(got.float().cpu(), ref, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("M,N,K", [
    (32, 4096, 4096),     # o_proj: cross-WG split path (slab + combine)
    (32, 12288, 4096),    # fused qkv: split=1, direct bf16 store
    (32, 4096, 11008),    # down_proj: split=4, k-step tail (688 % 16 != 0)
    (32, 22016, 4096),    # fused gate/up
    (17, 11008, 4096),    # M < 32 (clamped x rows dropped at epilogue)
    (1, 4096, 4096),      # single-sequence decode
    (32, 32000, 4096),    # lm_head
])
def test_decode_gemm(M, N, K):
    """csrc/decode_gemm.hip (v2 swizzled weight-stream kernel) vs fp32
    matmul, via the same swizzle helpers the serving path uses."""
    _assert_hip()
    torch.manual_seed(M * 31 + N)
    x = torch.randn(M, K, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(N, K, dtype=torch.bfloat16, device=DEV)
    ws = ops.ext().decode_swizzle_w(w)
    xs = ops.ext().decode_swizzle_x(x)
    y = ops.ext().decode_gemm(xs, ws, M, N, K)
    assert y.shape == (M, N) and y.dtype == torch.bfloat16
    ref = x.cpu().float() @ w.cpu().float().t()
    d = (y.cpu().float() - ref).abs().max().item()
    rel = d / ref.abs().max().item()
    assert rel < 2e-2, f"max abs {d} rel {rel}"


def test_decode_gemm_via_fast_linear():
    """fast_linear dispatches through the decode-weight registry and
    matches F.linear."""
    _assert_hip()
    from runbooks_amd.ops.linear import _DECODE_W_REGISTRY, \
        register_decode_weight
    torch.manual_seed(3)
    x = torch.randn(8, 4096, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(11008, 4096, dtype=torch.bfloat16, device=DEV)
    register_decode_weight(w)
    try:
        with torch.no_grad():
            y = ops.fast_linear(x, w)
        ref = torch.nn.functional.linear(x, w)
        d = (y.float() - ref.float()).abs().max() / ref.float().abs().max()
        assert d < 2e-2, d
    finally:
        _DECODE_W_REGISTRY.clear()


def test_decode_gemm_split_heuristic():
    """Split choice covers the 256 CUs on every flagship decode shape."""
    _assert_hip()
    e = ops.ext()
    for n, k in [(12288, 4096), (4096, 4096), (22016, 4096),
                 (4096, 11008), (32000, 4096)]:
        split = e.decode_gemm_split(n, k)
        assert (n // 32) * split >= 256, (n, k, split)
        assert (k // 16) % 1 == 0


@pytest.mark.parametrize("wt", [True, False])
def test_lora_delta(wt):
    """csrc/lora.hip fused LoRA merge vs torch addmm (both W layouts)."""
    _assert_hip()
    torch.manual_seed(5)
    T, r, N = 2048, 16, 4096
    t = torch.randn(T, r, dtype=torch.bfloat16, device=DEV)
    w = torch.randn((N, r) if wt else (r, N), dtype=torch.bfloat16,
                    device=DEV)
    y0 = torch.randn(T, N, dtype=torch.bfloat16, device=DEV)
    ref = (y0.float() + 0.5 * (t.float() @ (w.float().t() if wt
                                            else w.float()))).to(torch.bfloat16)
    y = y0.clone()
    ops.ext().lora_delta_(y, t, w, 0.5, wt)
    d = (y.float() - ref.float()).abs().max() / ref.float().abs().max()
    assert d < 2e-2, d


def test_lora_fused_train_step_matches_cpu_math():
    """One _LoRAFused fwd+bwd on GPU bf16 vs fp32 torch reference."""
    from runbooks_amd.train.lora import _LoRAFused
    torch.manual_seed(2)
    T, K, N, r, s = 256, 512, 1024, 16, 2.0
    x = torch.randn(T, K, dtype=torch.bfloat16, device=DEV,
                    requires_grad=True)
    w = torch.randn(N, K, dtype=torch.bfloat16, device=DEV)
    a = torch.randn(r, K, dtype=torch.bfloat16, device=DEV,
                    requires_grad=True)
    b = (torch.randn(N, r, dtype=torch.bfloat16, device=DEV) / 100
         ).requires_grad_()
    y = _LoRAFused.apply(x, w, a, b, s)
    dy = torch.randn_like(y)
    y.backward(dy)

    xf = x.detach().float().requires_grad_()
    af = a.detach().float().requires_grad_()
    bf = b.detach().float().requires_grad_()
    yf = xf @ w.float().t() + s * (xf @ af.t()) @ bf.t()
    yf.backward(dy.float())
    for got, ref, name in ((y, yf, "y"), (x.grad, xf.grad, "dx"),
                           (a.grad, af.grad, "da"), (b.grad, bf.grad, "db")):
        rel = (got.float() - ref).abs().max() / ref.abs().max().clamp(min=1e-6)
        assert rel < 5e-2, (name, rel)


def test_fp8_kv_append_and_decode():
    """fp8-e4m3 KV cache on GPU: kernel append vs CPU reference bytes,
    then paged decode over the fp8 cache vs the dequantized fp32 ref."""
    _assert_hip()
    from runbooks_amd.ops import kvcache as kc
    torch.manual_seed(1)
    B, hkv, G, bs, nblk, dh = 2, 4, 2, 16, 8, 128
    kcache, vcache = kc.alloc_kv_cache(nblk, hkv, dh, DEV, fp8=True)
    T = 40
    k = torch.randn(T, hkv, dh, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    ops.kv_append(k, v, kcache, vcache, slots)

    # reference append on CPU: dequantized caches must agree closely
    kr, vr = kc.alloc_kv_cache(nblk, hkv, dh, "cpu", fp8=True)
    kc.kv_append_ref(k.float().cpu(), v.float().cpu(), kr, vr, slots.cpu())
    dq_gpu = kc.fp8_dequant_cache_ref(kcache.cpu())
    dq_ref = kc.fp8_dequant_cache_ref(kr)
    # HIP's __hip_fp8_e4m3 and torch's converter may round a value one
    # e4m3 ulp apart (measured 2.9% of global max); the strict numerics
    # check is the decode comparison below, which dequantizes the SAME
    # GPU cache the kernel reads.
    rel = (dq_gpu - dq_ref).abs().max() / dq_ref.abs().max()
    assert rel < 6e-2, rel
    # and the original values are recovered within e4m3 row precision
    full = (dq_gpu.view(nblk * hkv * 16, dh)[:T * hkv]).reshape(-1)
    assert dq_gpu.abs().max() > 0

    # decode over the fp8 cache vs dequantized fp32 reference
    q = torch.randn(B, hkv * G, dh, dtype=torch.bfloat16, device=DEV)
    bt = torch.tensor([[0, 1], [2, 0]], dtype=torch.int32, device=DEV)
    sl = torch.tensor([23, 8], dtype=torch.int32, device=DEV)
    got = ops.paged_decode(q, kcache, vcache, bt, sl)
    ref = ops.paged_decode_ref(q.float().cpu(), kcache.cpu(), vcache.cpu(),
                               bt.cpu(), sl.cpu(),
                               scale=1.0 / math.sqrt(dh))
    d = (got.float().cpu() - ref).abs().max() / ref.abs().max()
    assert d < 3e-2, d


def test_fp8_kv_engine_gpu():
    """RB_KV_FP8 engine on GPU: generates valid tokens and auto-sizes
    ~2x the KV blocks of the bf16 cache."""
    _assert_hip()
    from runbooks_amd.models import build_model
    from runbooks_amd.serve import Engine
    m = build_model("smoke-llama", dtype=torch.bfloat16, device=DEV, seed=4)
    e8 = Engine(m, device=DEV, kv_blocks=128, seed=2, kv_fp8=True)
    out = e8.generate([3, 1, 4, 1, 5], max_new_tokens=8)
    assert len(out) == 8 and all(0 <= t < m.cfg.vocab_size for t in out)
    # capacity: fp8 blocks cost (dh+16)/2dh of bf16 bytes. Compare the
    # auto-sizing math directly (constructing two engines back to back
    # would let the first one's allocations shrink the second's budget).
    bf16_bpb = (2 * m.cfg.num_layers * m.cfg.num_kv_heads * e8.bs *
                m.cfg.head_dim * 2)
    fp8_bpb = (2 * m.cfg.num_layers * m.cfg.num_kv_heads * e8.bs *
               (m.cfg.head_dim + 16))
    assert fp8_bpb * 1.5 < bf16_bpb
    del e8
    torch.cuda.empty_cache()


def test_paged_decode_seq_starts():
    """Strict-window decode: kernel seq_starts vs the fp32 reference
    (split and non-split paths)."""
    _assert_hip()
    torch.manual_seed(9)
    B, hkv, G, bs, nblk, dh = 3, 2, 4, 16, 32, 128
    kc = torch.randn(nblk, hkv, bs, dh, dtype=torch.bfloat16, device=DEV)
    vc = torch.randn_like(kc)
    q = torch.randn(B, hkv * G, dh, dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(B * 8, dtype=torch.int32, device=DEV).reshape(B, 8)
    sl = torch.tensor([120, 77, 33], dtype=torch.int32, device=DEV)
    st = torch.tensor([88, 0, 17], dtype=torch.int32, device=DEV)
    ref = ops.paged_decode_ref(q.float().cpu(), kc.cpu(), vc.cpu(),
                               bt.cpu(), sl.cpu(),
                               scale=1.0 / math.sqrt(dh),
                               seq_starts=st.cpu())
    for nsplit in (1, 4):
        got = ops.paged_decode(q, kc, vc, bt, sl, nsplit=nsplit,
                               seq_starts=st)
        d = (got.float().cpu() - ref).abs().max() / ref.abs().max()
        assert d < 3e-2, (nsplit, d)
    # the same windows through the MFMA kernel (transposed-V layout —
    # the live config for mistral-style sliding windows at G>=4)
    vt = vc.permute(0, 1, 3, 2).contiguous()
    for nsplit in (1, 4):
        got = ops.paged_decode(q, kc, vt, bt, sl, nsplit=nsplit,
                               seq_starts=st)
        d = (got.float().cpu() - ref).abs().max() / ref.abs().max()
        assert d < 3e-2, ("vt", nsplit, d)


def test_paged_decode_with_operand_swz():
    """The fused o_proj operand emit matches decode_swizzle_x of the
    attention output."""
    _assert_hip()
    torch.manual_seed(4)
    B, hkv, G, bs, nblk, dh = 4, 8, 4, 16, 16, 128
    kc = torch.randn(nblk, hkv, bs, dh, dtype=torch.bfloat16, device=DEV)
    vc = torch.randn_like(kc)
    q = torch.randn(B, hkv * G, dh, dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(B * 4, dtype=torch.int32, device=DEV).reshape(B, 4)
    sl = torch.tensor([60, 33, 12, 7], dtype=torch.int32, device=DEV)
    # both kernel paths emit the operand: scalar (plain layout) and
    # MFMA (transposed-V layout)
    for v_dev in (vc, vc.permute(0, 1, 3, 2).contiguous()):
        for nsplit in (1, 4):
            out, swz = ops.paged_decode_with_operand(q, kc, v_dev, bt, sl,
                                                     nsplit=nsplit)
            assert swz is not None
            o2 = out.reshape(B, hkv * G * dh).contiguous()
            ref = ops.ext().decode_swizzle_x(o2)
            # rows m >= B are undefined in both layouts; compare live rows
            K = hkv * G * dh
            s_v = swz.view(K // 16, 2, 32, 8)
            r_v = ref.view(K // 16, 2, 32, 8)
            d = (s_v[:, :, :B].float() - r_v[:, :, :B].float()).abs().max()
            assert d == 0, (nsplit, d)


def test_flash_prefill_dh256():
    """gemma-width MFMA prefill (Dh=256) vs the fp32 chunked reference —
    the last eager inference fallback closed."""
    _assert_hip()
    torch.manual_seed(6)
    B, S, Hq, Hkv, DH = 2, 192, 4, 2, 256
    q = torch.randn(B, S, Hq, DH, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(B, S, Hkv, DH, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    got = ops.flash_prefill(q, k, v)
    ref = ops.causal_attention(q.float().cpu(), k.float().cpu(),
                               v.float().cpu())
    d = (got.float().cpu() - ref).abs().max() / ref.abs().max()
    assert d < 3e-2, d


@pytest.mark.parametrize("T,N", [(2048, 4096), (2048, 11008), (100, 352),
                                 (33, 4096)])
def test_lora_badd(T, N):
    """MFMA y += s * t[T,16] @ W[N,16]^T vs torch addmm."""
    _assert_hip()
    torch.manual_seed(T + N)
    y = torch.randn(T, N, dtype=torch.bfloat16, device=DEV)
    t = torch.randn(T, 16, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(N, 16, dtype=torch.bfloat16, device=DEV)
    ref = (y.float() + 2.0 * t.float() @ w.float().t())
    ops.ext().lora_badd_(y, t, w, 2.0)
    assert torch.allclose(y.float(), ref, atol=5e-2, rtol=5e-2), \
        (y.float() - ref).abs().max()


@pytest.mark.parametrize("hq,hkv,dh,nsplit", [(32, 8, 128, 1), (32, 8, 128, 4),
                                              (64, 4, 64, 1)])
def test_fp8_vt_mfma_decode(hq, hkv, dh, nsplit):
    """fp8-e4m3 transposed-V cache -> the fp8 MFMA decode kernel, append
    via the VT fp8 kernel, vs the dequantized fp32 reference."""
    _assert_hip()
    from runbooks_amd.ops import kvcache as kc
    from runbooks_amd.ops.attention import _is_vt
    torch.manual_seed(hq + dh)
    B, bs, nblk = 3, 16, 12
    kcache, vcache = kc.alloc_kv_cache(nblk, hkv, dh, DEV, fp8=True,
                                       v_transposed=True)
    assert _is_vt(kcache, vcache)
    T = 3 * 60
    k = torch.randn(T, hkv, dh, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    ops.kv_append(k, v, kcache, vcache, slots)

    q = torch.randn(B, hq, dh, dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(B * 4, dtype=torch.int32, device=DEV).reshape(B, 4)
    sl = torch.tensor([60, 47, 12], dtype=torch.int32, device=DEV)
    st = torch.tensor([5, 0, 0], dtype=torch.int32, device=DEV)
    got = ops.paged_decode(q, kcache, vcache, bt, sl, nsplit=nsplit,
                           seq_starts=st)
    ref = ops.paged_decode_ref(q.float().cpu(), kcache.cpu(), vcache.cpu(),
                               bt.cpu(), sl.cpu(),
                               scale=1.0 / math.sqrt(dh),
                               seq_starts=st.cpu())
    d = (got.float().cpu() - ref).abs().max() / ref.abs().max()
    assert d < 3e-2, d


def test_fp8_vt_append_matches_plain_layout():
    """VT fp8 append stores the same dequantized values as the plain
    fp8 layout."""
    _assert_hip()
    from runbooks_amd.ops import kvcache as kc
    torch.manual_seed(2)
    hkv, dh, nblk, T = 4, 128, 4, 30
    k = torch.randn(T, hkv, dh, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    k1, v1 = kc.alloc_kv_cache(nblk, hkv, dh, DEV, fp8=True)
    k2, v2 = kc.alloc_kv_cache(nblk, hkv, dh, DEV, fp8=True,
                               v_transposed=True)
    ops.kv_append(k, v, k1, v1, slots)
    ops.kv_append(k, v, k2, v2, slots)
    assert torch.equal(k1, k2)
    d1 = kc.fp8_dequant_cache_ref(v1.cpu())           # [nb,hkv,bs,dh]
    d2 = kc.fp8_dequant_cache_ref(v2.cpu())           # [nb,hkv,dh,bs]
    assert torch.allclose(d1, d2.permute(0, 1, 3, 2), atol=1e-6)


@pytest.mark.parametrize("T", [1, 15, 33, 129, 300])
@pytest.mark.parametrize("K,widths", [(64, (64,)), (192, (128, 64)),
                                      (704, (256, 64, 64))])
def test_lora_siblings(T, K, widths):
    """Products of rank-16 adapters side by side vs fp64: sums in fp32, one
    rounding to bf16 (2^-9 of a value, half of that over many)."""
    _assert_hip()
    ext = ops.ext()
    torch.manual_seed(T + K)
    x, *A = (torch.randn(n, K, device=DEV).bfloat16()
             for n in (T, *[16] * len(widths)))
    B = [torch.randn(n, 16, device=DEV).bfloat16() for n in widths]
    y = torch.randn(T, sum(widths), device=DEV).bfloat16()

    def close(got, ref):
        assert (got.double() - ref).norm() < 2 ** -8 * ref.norm()

    xd, ys = x.double(), y.double().split(widths, 1)
    Ad, Bd = [a.double() for a in A], [b.double() for b in B]
    t, dt = ext.lora_down(x, A), ext.lora_down_columns(y, B, 2.0)
    close(t, torch.stack([xd @ a.t() for a in Ad]))
    close(dt, torch.stack([2 * v @ b for v, b in zip(ys, Bd)]))
    td, dtd = t.double(), dt.double()
    y2, x2 = y.clone(), x.clone()
    ext.lora_add_(y2, t, B, 2.0, False)
    ext.lora_add_(x2, dt, A, 1.0, True)
    close(y2, y.double() + 2 * torch.cat([v @ b.t() for v, b in
                                          zip(td, Bd)], 1))
    close(x2, xd + sum(d @ a for d, a in zip(dtd, Ad)))
    close(ext.lora_grad(y, t, list(widths), 2.0, False),
          torch.cat([2 * v.t() @ u for v, u in zip(ys, td)]))
    close(ext.lora_grad(x, dt, [], 1.0, True),
          torch.cat([d.t() @ xd for d in dtd]))


@pytest.mark.parametrize("T", [1, 17, 130])
@pytest.mark.parametrize("K,widths", [
    (1088, (1088,)),            # a last chunk by itself, waves without one
    (2048, (2112, 64)),         # as many chunks as are fetched ahead
    (8256, (4160, 64, 1024))])  # many turns
def test_lora_siblings_long(T, K, widths):
    """Sums over more columns than all waves fetch at a time, and both gradients
    in one launch, which are the same as each by itself."""
    _assert_hip()
    ext = ops.ext()
    torch.manual_seed(T + K)
    x, *A = (torch.randn(n, K, device=DEV).bfloat16()
             for n in (T, *[16] * len(widths)))
    B = [torch.randn(n, 16, device=DEV).bfloat16() for n in widths]
    y = torch.randn(T, sum(widths), device=DEV).bfloat16()
    t, dt = ext.lora_down(x, A), ext.lora_down_columns(y, B, 2.0)
    # fp32 sums and one rounding
    for got, ref in ((t, [x.double() @ a.double().t() for a in A]),
                     (dt, [2 * v.double() @ b.double() for v, b in
                           zip(y.split(widths, 1), B)])):
        ref = torch.stack(ref)
        assert (got.double() - ref).norm() < 2 ** -8 * ref.norm()
    db, da = ext.lora_grads(y, t, x, dt, list(widths), 2.0)
    assert torch.equal(db, ext.lora_grad(y, t, list(widths), 2.0, False))
    assert torch.equal(da, ext.lora_grad(x, dt, [], 1.0, True))


@pytest.mark.parametrize("heads,kv,dh,B,S", [(4, 4, 64, 2, 33),
                                             (4, 1, 128, 1, 100),
                                             (6, 2, 64, 3, 1)])
def test_lora_siblings_train(heads, kv, dh, B, S, monkeypatch):
    """Loss and gradients with the siblings' results side by side: no further
    from fp32 than with every adapter by itself, up to the chance of rounding."""
    _assert_hip()
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer
    from runbooks_amd.train.lora import apply_lora

    cfg = ModelConfig("siblings", 256, heads * dh, 2, heads, kv, 320,
                      max_seq_len=128, head_dim=dh)
    tokens = torch.randint(0, 256, (B, S + 1),
                           generator=torch.Generator().manual_seed(S))

    def run(dtype, device, one_by_one=False):
        monkeypatch.setenv("RB_LORA_MFMA", "0" if one_by_one else "1")
        torch.manual_seed(3)
        m = Transformer(cfg, dtype=torch.bfloat16).to(device)
        for p in m.parameters():
            p.data = p.data.to(dtype)
        for p in m.parameters():
            if p.dim() == 2:        # the same everywhere, exact in bf16
                p.data = (p.data.float() * 4).bfloat16().to(p)
        apply_lora(m, r=16, alpha=32)
        g = torch.Generator().manual_seed(4)
        for n, p in m.named_parameters():
            if "lora" in n:
                p.data = (torch.randn(p.shape, generator=g) * 0.05) \
                    .bfloat16().to(p)
        logits = m(tokens[:, :-1].to(device))
        loss = torch.nn.functional.cross_entropy(
            logits.float().view(-1, 256), tokens[:, 1:].reshape(-1).to(device))
        loss.backward()
        return [loss.detach().float().cpu().view(1)] + [
            p.grad.float().cpu() for n, p in m.named_parameters()
            if "lora" in n]

    ref = run(torch.float32, "cpu")
    new = run(torch.bfloat16, DEV)
    old = run(torch.bfloat16, DEV, one_by_one=True)

    def far(got):
        return sum(((g - r).norm() / (r.norm() + 1e-6)) ** 2
                   for g, r in zip(got[1:], ref[1:])).sqrt()

    assert abs(new[0] - ref[0]) < 2e-2 * ref[0]
    assert far(new) < 1.25 * far(old) + 1e-3


@pytest.mark.parametrize("rows,n,k", [(1281, 2816, 64), (2048, 11008, 64),
                                      (1536, 10816, 192), (300, 192, 8192),
                                      (129, 16448, 64), (257, 16512, 4096),
                                      (65, 32768, 64), (65, 32832, 64)])
def test_wide_products(rows, n, k):
    """Products in one or two calls, [rows, k] by [n, k] and back, vs fp64."""
    from runbooks_amd.ops.linear import wide_product, wide_product_grad
    torch.manual_seed(rows)
    x = torch.randn(rows, k, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16()
    y = torch.randn(rows, n, device=DEV).bfloat16()
    for got, ref in ((wide_product(x, w), x.double() @ w.double().t()),
                     (wide_product_grad(x, w.t().contiguous()),
                      x.double() @ w.double().t()),
                     (wide_product_grad(y, w), y.double() @ w.double())):
        # one rounding of the result (at most 2^-9 of each value; of two the
        # norm is larger, 2^-8.9), fp32 sums
        assert (got.double() - ref).norm() < (2 ** -9 + 1e-5) * ref.norm()


@pytest.mark.parametrize("rows,n,k", [
    (20, 10240, 1024),              # a registered copy that shares x
    (1400, 4096, 1024),             # tiles
    (2048, 3584, 8256),             # one round of tiles
    (1536, 11008, 64)])             # two calls
@pytest.mark.parametrize("which", ["x", "weight"])
def test_wide_products_are_differentiated(rows, n, k, which):
    """Gradients of what wide_linear and wide_product return, whichever way the
    product would take without them: one rounding, fp32 sums."""
    from runbooks_amd.ops.linear import (register_decode_weight, wide_linear,
                                         wide_product)
    torch.manual_seed(rows)
    x = torch.randn(rows, k, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16()
    dy = torch.randn(rows, n, device=DEV).bfloat16()
    if rows <= 32:
        register_decode_weight(w)
    (x if which == "x" else w).requires_grad_()
    want = dy.double() @ w.double() if which == "x" else \
        dy.double().t() @ x.double()
    ref = x.detach().double() @ w.detach().double().t()
    for product in (wide_linear, wide_product):
        y = product(x, w)
        assert (y.double() - ref).norm() < 2 ** -8 * ref.norm()
        got, = torch.autograd.grad(y, x if which == "x" else w, dy)
        assert (got.double() - want).norm() < 2 ** -8 * want.norm()


@pytest.mark.parametrize("rows,n,k,halves", [
    (20, 16448, 64, True), (2304, 17408, 4096, True), (300, 32768, 60, True),
    (20, 16384, 64, False), (20, 32832, 64, False), (20, 16448, 62, False)])
def test_long_sums_of_input_gradients(monkeypatch, rows, n, k, halves):
    """Sums that are left to the library and long go in two fp32 halves, rounded
    once: on either side of the rule."""
    from runbooks_amd.ops import linear
    torch.manual_seed(rows)
    dy = torch.randn(rows, n, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16()
    summed, sum_parts = [], ops.ext().sum_parts
    monkeypatch.setattr(ops.ext(), "sum_parts",
                        lambda p: summed.append(p.shape) or sum_parts(p))
    got = linear.wide_product_grad(dy, w)
    assert summed == ([(2, rows, k)] if halves else [])
    ref = dy.double() @ w.double()
    assert (got.double() - ref).norm() < (2 ** -9 + 1e-5) * ref.norm()


@pytest.mark.parametrize("M", [1, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("N,K", [(32, 1024), (96, 1040), (20512, 1024),
                                 (160, 8208), (4096, 4096)])
def test_decode_gemm_rows(M, N, K):
    """Rows as they are by a weight in the decode layout vs fp64: one rounding
    of the result."""
    _assert_hip()
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = torch.randn(N, K, device=DEV).bfloat16()
    y = ops.ext().decode_gemm_rows(x, ops.ext().decode_swizzle_w(w), N)
    ref = x.double() @ w.double().t()
    assert (y.double() - ref).norm() < 2 ** -8 * ref.norm()


@pytest.mark.parametrize("m", [1, 16, 20, 32, 40])
@pytest.mark.parametrize("fp8", [False, True])
def test_products_of_changed_weight(m, fp8):
    """Products of any number of rows follow a weight that changes in place,
    whichever of its layouts they would read."""
    from runbooks_amd.ops.linear import (decode_linear_raw, fast_linear,
                                         quantize_fp8, register_decode_weight,
                                         wide_linear)
    torch.manual_seed(m)
    w = torch.randn(10240, 1024, device=DEV).bfloat16()
    x = torch.randn(m, 1024, device=DEV).bfloat16()
    (quantize_fp8 if fp8 else register_decode_weight)(w)
    products = [fast_linear, wide_linear]
    if m <= 32:
        products.append(lambda x, w: decode_linear_raw(x, w)[0])
    with torch.no_grad():
        w.copy_(torch.randn(10240, 1024, device=DEV))
        ref = x.double() @ w.double().t()
        for product in products:
            y = product(x, w).double()
            y = y.sum(0) if y.dim() == 3 else y
            assert (y - ref).norm() < 2 ** -8 * ref.norm()


@pytest.mark.parametrize("m", [1, 40])
@pytest.mark.parametrize("uniform", [True, False])
def test_products_of_trained_weight(m, uniform):
    """A step of the optimizer, whose kernels write past autograd, is followed
    by the products of a weight that has a decode layout."""
    from runbooks_amd.ops.linear import fast_linear, register_decode_weight
    torch.manual_seed(m)
    w = torch.nn.Parameter(torch.randn(64, 1024, device=DEV).bfloat16())
    other = torch.nn.Parameter(torch.ones(8, device=DEV).bfloat16())
    register_decode_weight(w)
    opt = ops.FusedAdamW([w, other], lr=0.1)
    if not uniform:             # a step for each parameter
        other.grad = torch.ones_like(other)
        opt.step()
    other.grad, w.grad = torch.ones_like(other), torch.randn_like(w)
    opt.step()
    x = torch.randn(m, 1024, device=DEV).bfloat16()
    with torch.no_grad():
        y = fast_linear(x, w)
    ref = x.double() @ w.double().t()
    assert (y - ref).norm() < 2 ** -8 * ref.norm()


def test_decode_gemm_rows_of_changed_weight():
    """Products of 33 to 128 rows follow a weight that changes in place."""
    from runbooks_amd.ops.linear import fast_linear, register_decode_weight
    w = torch.randn(64, 1024, device=DEV).bfloat16()
    x = torch.randn(40, 1024, device=DEV).bfloat16()
    register_decode_weight(w)
    with torch.no_grad():
        before = fast_linear(x, w)
        w.mul_(2)
        after = fast_linear(x, w)
    assert (after - 2 * before).norm() < 2 ** -7 * after.norm()


@pytest.mark.parametrize("m,n,k", [(33, 64, 16448), (700, 260, 24576)])
def test_long_rows(m, n, k):
    """Sums in two fp32 parts: one rounding of the result, as in one."""
    from runbooks_amd.ops.linear import fast_linear
    torch.manual_seed(m)
    x = torch.randn(m, k, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16()
    with torch.no_grad():
        y = fast_linear(x, w)
    ref = x.double() @ w.double().t()
    assert (y.double() - ref).norm() < 2 ** -8 * ref.norm()



@pytest.mark.parametrize("hq,hkv,dh,vt", [(3, 3, 64, False), (16, 4, 64, False),
                                          (16, 1, 64, False), (8, 2, 128, False),
                                          (8, 2, 64, True), (4, 4, 256, False)])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_paged_decode_operand(hq, hkv, dh, vt, nsplit):
    """The operand that goes with the result holds the same values, whatever a
    lane's share of a head."""
    _assert_hip()
    from runbooks_amd.ops import kvcache as kc
    torch.manual_seed(hq + dh)
    B = 5
    k, v = kc.alloc_kv_cache(B * 4, hkv, dh, DEV, v_transposed=vt)
    k.normal_()
    v.normal_()
    q = torch.randn(B, hq, dh, dtype=torch.bfloat16, device=DEV)
    bt = torch.arange(B * 4, dtype=torch.int32, device=DEV).view(B, 4)
    sl = torch.tensor([64, 1, 17, 33, 50], dtype=torch.int32, device=DEV)
    out, swz = ops.paged_decode_with_operand(q, k, v, bt, sl, nsplit=nsplit)
    rows = swz.view(-1, 2, 32, 8)[:, :, :B].permute(2, 0, 1, 3)
    assert torch.equal(rows.reshape(B, hq * dh), out.view(B, hq * dh))


@pytest.mark.parametrize("B", [1, 7, 32])
@pytest.mark.parametrize("act,bias,ff", [("relu", True, 352),
                                         ("gelu_tanh", True, 1056),
                                         ("gelu", False, 64)])
def test_decode_affine(B, act, bias, ff, monkeypatch):
    """Decode of layer-norm models in nine launches a layer: no further from
    fp32 than in launches of their own."""
    _assert_hip()
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer, fuse_for_inference
    cfg = ModelConfig("affine", 256, 192, 2, 3, 3, ff, max_seq_len=128,
                      head_dim=64, norm="layernorm", act=act, pos="learned",
                      attn_bias=bias, mlp_bias=bias)
    g = torch.Generator().manual_seed(B)
    lens = torch.randint(1, 60, (B,), generator=g)
    tokens = torch.randint(0, 256, (B,), generator=g)
    tables = torch.arange(B * 4).view(B, 4)
    kv = [torch.randn(B * 4, 3, 16, 64, generator=g).bfloat16()
          for _ in range(4)]
    slots = torch.tensor([int(tables[i, (n - 1) // 16]) * 16 + (n - 1) % 16
                          for i, n in enumerate(lens.tolist())])

    def run(dtype, device):
        torch.manual_seed(1)
        m = Transformer(cfg, dtype=torch.bfloat16).to(device)
        with torch.no_grad():
            for p in m.parameters():
                p.data = p.data.to(dtype)
                if p.dim() == 1:
                    p += torch.linspace(-0.5, 0.5, p.numel(),
                                        device=device).bfloat16().to(dtype)
        if device != "cpu":
            fuse_for_inference(m.eval())
        caches = [tuple(c.to(device, dtype, copy=True) for c in kv[i:i + 2])
                  for i in (0, 2)]
        i32 = dict(device=device, dtype=torch.int32)
        out = m.decode(tokens.to(device), (lens - 1).to(**i32), caches,
                       slots.to(**i32), tables.to(**i32), lens.to(**i32),
                       nsplit=1)
        return m, out.float().cpu(), [c.float().cpu() for kc in caches
                                      for c in kc]

    _, ref, ref_kv = run(torch.float32, "cpu")
    m, new, new_kv = run(torch.bfloat16, DEV)
    assert m._affine_ready()
    monkeypatch.setenv("RB_FUSED_RESID", "0")
    _, old, old_kv = run(torch.bfloat16, DEV)

    def far(got, want):
        return ((got - want).norm() / want.norm()).item()

    assert far(new, ref) < 1.1 * far(old, ref) + 1e-3
    for n, o, r in zip(new_kv, old_kv, ref_kv):
        assert far(n, r) < 1.1 * far(o, r) + 1e-4
    with torch.no_grad():       # weights that change leave the path
        m.blocks[0].mlp.fc1.weight.mul_(2)
    assert not m._affine_ready()


@pytest.mark.parametrize("B,S", [(1, 1), (2, 63), (3, 65)])
def test_layer_norm_sums(B, S):
    """Logits of a layer-norm model with the residual's sums in the norms and
    biases in the products: no further from fp32 than without."""
    _assert_hip()
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer
    cfg = ModelConfig("sums", 256, 192, 2, 3, 3, 352, max_seq_len=128,
                      head_dim=64, norm="layernorm", act="relu", pos="learned",
                      attn_bias=True, mlp_bias=True)
    tokens = torch.randint(0, 256, (B, S),
                           generator=torch.Generator().manual_seed(S))

    def run(dtype, device, grad):
        torch.manual_seed(1)
        m = Transformer(cfg, dtype=torch.bfloat16).to(device)
        for p in m.parameters():
            p.data = p.data.to(dtype)
            if p.dim() == 1:
                p.data += torch.linspace(-0.5, 0.5, p.numel(),
                                         device=device).bfloat16().to(dtype)
        with torch.set_grad_enabled(grad):
            return m(tokens.to(device)).detach().float().cpu()

    ref = run(torch.float32, "cpu", False)
    new, old = run(torch.bfloat16, DEV, False), run(torch.bfloat16, DEV, True)
    assert (new - ref).norm() < 1.1 * (old - ref).norm() + 1e-3 * ref.norm()


@pytest.mark.parametrize("M,widths,K", [
    (1, [32], 32), (16, [32, 64, 32], 96), (17, [64, 32, 32], 288),
    (31, [4096], 160), (32, [4128], 1056), (9, [4128, 32], 800)])
@pytest.mark.parametrize("act,bias", [(0, True), (1, False), (2, True),
                                      (3, True)])
def test_decode_affine_products(M, widths, K, act, bias):
    """Edges of the row blocks, of the waves' shares of K and of the matrices;
    fp32 sums, one rounding (2^-9 relative, twice that for the sums' own and
    the activation's)."""
    _assert_hip()
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    ws = [torch.randn(n, K, generator=g, device=DEV).bfloat16()
          for n in widths]
    bs = [torch.randn(n, generator=g, device=DEV).bfloat16() if bias else None
          for n in widths]
    xs = ops.ext().decode_swizzle_x(x)
    out = ops.ext().decode_affine(xs, ws, bs, M, act)
    f = [lambda y: y, torch.relu, torch.nn.functional.gelu,
         lambda y: torch.nn.functional.gelu(y, approximate="tanh")][act]
    for y, w, b in zip(out, ws, bs):
        ref = x.double() @ w.double().t()
        ref = f(ref if b is None else ref + b.double())
        assert y.shape == ref.shape
        assert (y - ref).norm() <= 2 ** -8 * ref.norm()
    h = ops.ext().decode_affine(xs, ws[:1], bs[:1], M, act, operand=True)[0]
    assert torch.equal(h.view(-1, 2, 32, 8)[:, :, :M].permute(2, 0, 1, 3)
                       .reshape(M, -1), out[0])


@pytest.mark.parametrize("batch", [1, 20])
@pytest.mark.parametrize("name", ["q_proj", "v_proj.bias", "fc1", "fc1.bias",
                                  "o_proj", "down_proj.bias"])
def test_captured_decode_follows_weights(name, batch):
    """A captured step of a layer-norm model computes with weights that were
    changed after the capture, as an eager one does: through the parameter, or
    past its version through .data."""
    _assert_hip()
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer, fuse_for_inference
    from runbooks_amd.serve.graph import GraphedDecoder
    cfg = ModelConfig("follow", 256, 192, 2, 3, 3, 352, max_seq_len=64,
                      head_dim=64, norm="layernorm", act="relu", pos="learned",
                      attn_bias=True, mlp_bias=True)
    torch.manual_seed(1)
    m = fuse_for_inference(Transformer(cfg, dtype=torch.bfloat16, tp=1)
                           .to(DEV).eval())
    caches = m.alloc_caches(batch + 1, DEV)
    for c in (c for kv in caches for c in kv):
        c.normal_()
    step = (list(range(batch)), [9] * batch,
            [i * 16 + 9 for i in range(batch)], [[i] for i in range(batch)],
            [10] * batch)
    i32 = dict(device=DEV, dtype=torch.int32)

    def eager():
        return m.decode(torch.tensor(step[0], device=DEV),
                        torch.tensor(step[1], **i32), caches,
                        torch.tensor(step[2], **i32),
                        torch.tensor(step[3], **i32),
                        torch.tensor(step[4], **i32), nsplit=1)

    with torch.no_grad():
        graphed = GraphedDecoder(m, caches, batch, 1, batch, DEV)
        layer, _, which = name.partition(".")
        blk = m.blocks[1]
        p = getattr(getattr(blk.attn, layer, None) or getattr(blk.mlp, layer),
                    which or "weight")
        before = graphed.decode(*step).clone()
        assert m._affine_ready()
        for change in (p, p.data):
            change.add_(torch.randn_like(p))
            got, want = graphed.decode(*step), eager()
            assert (got - want).norm() < 0.02 * want.norm()
            assert (got - before).norm() > 0.05 * before.norm()
            before = got.clone()


@pytest.mark.parametrize("batch", [1, 20, 40])
@pytest.mark.parametrize("eight_bit", [False, True])
def test_captured_decode_follows_weights_with_copies(batch, eight_bit):
    """A captured step whose products read copies of the weights is captured
    again once a weight has been written to."""
    _assert_hip()
    from runbooks_amd.models.config import ModelConfig
    from runbooks_amd.models.transformer import Transformer, fuse_for_inference
    from runbooks_amd.serve.graph import GraphedDecoder
    cfg = ModelConfig("copies", 256, 1024, 2, 8, 8, 1024, max_seq_len=64,
                      head_dim=128)
    torch.manual_seed(1)
    m = fuse_for_inference(Transformer(cfg, dtype=torch.bfloat16, tp=1)
                           .to(DEV).eval(), load_in_8bit=eight_bit)
    caches = m.alloc_caches(batch + 1, DEV)
    for c in (c for kv in caches for c in kv):
        c.normal_()
    step = (list(range(batch)), [9] * batch,
            [i * 16 + 9 for i in range(batch)], [[i] for i in range(batch)],
            [10] * batch)
    i32 = dict(device=DEV, dtype=torch.int32)
    with torch.no_grad():
        graphed = GraphedDecoder(m, caches, batch, 1, batch, DEV)
        before = graphed.decode(*step).clone()
        first = graphed.graphs[batch][0]
        for p in (m.blocks[1].attn.v_proj.weight, m.blocks[0].mlp.up_proj.weight,
                  m.blocks[1].mlp.down_proj.weight, m.lm_head.weight):
            graphed.decode(*step)
            assert graphed.graphs[batch][0] is first
            p.copy_(torch.randn_like(p) * 0.05)
            got = graphed.decode(*step).clone()
            want = m.decode(torch.tensor(step[0], device=DEV),
                            torch.tensor(step[1], **i32), caches,
                            torch.tensor(step[2], **i32),
                            torch.tensor(step[3], **i32),
                            torch.tensor(step[4], **i32), nsplit=1)
            assert (got - want).norm() < 0.02 * want.norm()
            assert (got - before).norm() > 0.05 * before.norm()
            before, first = got, graphed.graphs[batch][0]


@pytest.mark.parametrize("where", ["block", "norm1", "fc1", "adapters"])
def test_decode_affine_leaves_modules_that_do_more(where):
    """A hook, or an adapter put in later, takes decoding off the path that
    does the work of its module."""
    _assert_hip()
    from runbooks_amd.models import build_model
    from runbooks_amd.models.transformer import fuse_for_inference
    from runbooks_amd.train import apply_lora
    m = fuse_for_inference(build_model("opt-125m", dtype=torch.bfloat16, tp=1,
                                       device=DEV).eval())
    caches = m.alloc_caches(2, DEV)
    i32 = dict(device=DEV, dtype=torch.int32)

    def decode():
        return m.decode(torch.tensor([5], device=DEV),
                        torch.tensor([0], **i32), caches,
                        torch.tensor([0], **i32), torch.tensor([[0]], **i32),
                        torch.tensor([1], **i32), nsplit=1)

    first = decode()
    assert m._affine_ready()
    blk, fired = m.blocks[1], []
    if where == "adapters":
        apply_lora(m, r=8)
        with torch.no_grad():
            blk.mlp.fc1.lora_b.normal_()
        assert not torch.allclose(decode(), first, atol=1e-2)
        return
    {"block": blk, "norm1": blk.norm1, "fc1": blk.mlp.fc1}[
        where].register_forward_hook(lambda *a: fired.append(1))
    again = decode()
    assert fired == [1]
    assert (again - first).norm() < 0.03 * first.norm()


@pytest.mark.parametrize("name", ["opt-125m", "smoke-llama"])
def test_prefill_hooks_fire(name):
    _assert_hip()
    from runbooks_amd.models import build_model
    m = build_model(name, dtype=torch.bfloat16, tp=1, device=DEV).eval()
    tokens, fired = torch.arange(40, device=DEV).view(1, 40), []
    with torch.no_grad():
        want = m(tokens)
        for mod in (m.blocks[0], m.blocks[1].norm2, m.norm_f):
            mod.register_forward_hook(lambda *a: fired.append(1))
        got = m(tokens)
    assert len(fired) == 3
    assert (got - want).norm() < 0.03 * want.norm()


def test_fp8_decode_takes_positions_of_64_bits():
    """As rotation and append in launches of their own did."""
    _assert_hip()
    from runbooks_amd.models import build_model
    from runbooks_amd.models.transformer import fuse_for_inference
    m = fuse_for_inference(build_model("smoke-llama", dtype=torch.bfloat16,
                                       tp=1, device=DEV).eval())
    caches = m.alloc_caches(4, DEV, fp8=True)
    for c in (c for kv in caches for c in kv):
        c.zero_()
    i32 = dict(device=DEV, dtype=torch.int32)

    def decode(dtype):
        return m.decode(torch.tensor([3, 5], device=DEV),
                        torch.tensor([0, 0], device=DEV, dtype=dtype), caches,
                        torch.tensor([0, 16], device=DEV, dtype=dtype),
                        torch.tensor([[0], [1]], **i32),
                        torch.tensor([1, 1], **i32), nsplit=1)

    assert torch.equal(decode(torch.int64), decode(torch.int32))


@pytest.mark.parametrize("narrow", [32, 64])
def test_lora_siblings_of_other_widths(narrow):
    """Sibling adapters of which some could run on the packed kernels and
    others not: every pass uses its own input, and nothing of it stays."""
    _assert_hip()
    from runbooks_amd.train.lora import apply_lora
    torch.manual_seed(0)
    net = torch.nn.Module()
    for name, n in (("q_proj", 64), ("k_proj", narrow), ("v_proj", narrow)):
        setattr(net, name, torch.nn.Linear(64, n, bias=False))
    net = net.to(DEV, torch.bfloat16)
    apply_lora(net, r=16)
    members = [net.q_proj, net.k_proj, net.v_proj]
    with torch.no_grad():
        for m in members:
            m.lora_b.normal_()
    for _ in range(4):
        x = torch.randn(40, 64, device=DEV).bfloat16()
        for m in members:
            ref = x.double() @ (m.weight.double().t() + m.scale *
                                m.lora_a.double().t() @ m.lora_b.double().t())
            # t and the result are rounded, the latter twice at most
            assert (m(x) - ref).norm() < 2 ** -7 * ref.norm()
        assert m._group._t is None
        del x


def test_lora_packed_takes_any_gradient():
    """A gradient that starts off a 16-byte boundary."""
    _assert_hip()
    from runbooks_amd.train.lora import LoRALinear
    torch.manual_seed(0)
    layer = LoRALinear(torch.nn.Linear(64, 128, bias=False).to(
        DEV, torch.bfloat16), r=16)
    with torch.no_grad():
        layer.lora_b.normal_()
    x = torch.randn(40, 64, device=DEV).bfloat16().requires_grad_()
    dy = torch.randn(40 * 128 + 1, device=DEV).bfloat16()[1:].view(40, 128)
    grads = [torch.autograd.grad(layer(x), (x, layer.lora_a, layer.lora_b), g)
             for g in (dy, dy.clone())]
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("T", [1, 63, 130, 256])
@pytest.mark.parametrize("transposed", [False, True])
def test_lora_grad_of_infinite_rows(T, transposed):
    """An infinite value in the last row is infinite in its column's sums, and
    in no other's."""
    _assert_hip()
    torch.manual_seed(T)
    x = torch.randn(T, 128, device=DEV).bfloat16()
    x[-1, 70] = float("inf")
    t = torch.randn(2, T, 16, device=DEV).bfloat16()
    got = ops.ext().lora_grad(x, t, [64, 64], 1.0, transposed).double()
    if transposed:
        ref = torch.cat([m.double().t() @ x.double() for m in t])
    else:
        ref = torch.cat([x[:, i * 64:i * 64 + 64].double().t() @ t[i].double()
                         for i in range(2)])
    assert torch.equal(got.isinf(), ref.isinf()) and not got.isnan().any()
    assert torch.equal(got.sign()[got.isinf()], ref.sign()[ref.isinf()])
    assert ((got - ref)[ref.isfinite()].norm() <
            2 ** -8 * ref[ref.isfinite()].norm())
