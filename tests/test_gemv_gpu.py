"""``ome_gemv`` (batch-1..8 weight-streaming GEMV, ``csrc/kernels/gemv.hip``) vs an fp32 PyTorch
reference: every row count, N not a multiple of the 16-row workgroup span, K tails below one
512-element step, bias, strided activations and output."""
import pytest
import torch

from ome_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(4096, 4096), (6144, 4096), (4096, 14336), (1000, 1032), (37, 200), (16, 8),
                                 (2048, 2560)])
def test_gemv_matches_reference(M, N, K):
    torch.manual_seed(0)
    xs = torch.randn(M, K + 64, device="cuda").to(torch.bfloat16)
    x = xs[:, 16:16 + K]
    w = (torch.randn(N, K, device="cuda") * 0.05).to(torch.bfloat16)
    b = (torch.randn(N, device="cuda") * 0.1).to(torch.bfloat16)
    want = x.float() @ w.float().t()
    big = torch.full((M, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)
    for bias in (None, b):
        ref = want if bias is None else want + b.float()
        got = ops.gemv(x, w, bias, out=big[:, :N]).float()
        assert (got - ref).abs().max().item() < 1e-2 * max(1.0, ref.abs().max().item())
        assert (big[:, N:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,I", [(4096, 14336), (2048, 8192), (1024, 512)])
def test_gemv_act_equals_act_then_gemv(M, N, I):
    """Down projection with SwiGLU folded into the operand load: bit-identical to act_and_mul
    followed by the plain GEMV (same bf16 rounding of the activation), close to fp32."""
    from ome_amd import ops
    from ome_amd.ops import reference as ref

    torch.manual_seed(M * 7 + N)
    gu = torch.randn(M, 2 * I, device="cuda", dtype=torch.bfloat16) * 2
    w = torch.randn(N, I, device="cuda", dtype=torch.bfloat16) * 0.05
    fused = ops.gemv_act(gu, w)
    two = ops.gemv(ops.act_and_mul(gu, 0), w)
    assert torch.equal(fused, two)
    want = torch.nn.functional.linear(ref.act_and_mul(gu.float().cpu(), 0), w.float().cpu())
    assert torch.allclose(fused.float().cpu(), want, atol=2e-2 * want.abs().max().item(), rtol=2e-2)


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("I,K", [(14336, 4096), (2048, 8192), (2064, 1032), (48, 200), (16, 8)])
def test_gemv_swiglu_equals_gemv_then_act(M, I, K):
    torch.manual_seed(M + I)
    x = torch.randn(M, K + 8, device="cuda").to(torch.bfloat16)[:, 8:]
    w = (torch.randn(2 * I, K, device="cuda") / K ** 0.5).to(torch.bfloat16)
    assert torch.equal(ops.gemv_swiglu(x, w), ops.act_and_mul(ops.gemv(x, w), 0, interleaved=True))


@pytest.mark.parametrize("M", [1, 3, 4, 8])
@pytest.mark.parametrize("Hq,Hkv,D,K", [(32, 8, 128, 4096), (3, 1, 64, 72), (2, 2, 256, 8192), (4, 1, 128, 1032)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2], ids=str)
def test_gemv_qkv_equals_gemv_then_rope(M, Hq, Hkv, D, K, cache):
    torch.manual_seed(M + D)
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, device="cuda") / K ** 0.5).to(torch.bfloat16)
    bias = torch.randn(w.shape[0], device="cuda").to(torch.bfloat16) if M % 2 else None
    ang = torch.rand(50, D // 2, device="cuda") * 6
    cs = torch.cat([ang.cos(), ang.sin()], 1).contiguous()
    pos = torch.randint(0, 50, (M,), dtype=torch.int32, device="cuda")
    slots = torch.randperm(5 * 16, device="cuda")[:M].int()
    if M > 3:
        slots[2] = -1   # a padded row: no cache write
    new = lambda *s: (torch.randn(*s, device="cuda") * 0.5).to(cache)  # noqa: E731
    kc, vc = new(5, Hkv, 16, D), new(5, Hkv, D, 16)
    k2, v2, q1 = kc.clone(), vc.clone(), torch.empty(M, Hq, D, dtype=torch.bfloat16, device="cuda")
    q2, sc = torch.empty_like(q1), (1.0, 1.0) if cache == torch.bfloat16 else (0.5, 2.0)
    assert ops.gemv_qkv_ok(x, w, bias, D, D, Hq, Hkv, kc)
    ops.gemv_qkv(x, w, bias, pos, cs, q1, kc, vc, slots, Hq, Hkv, D, *sc)
    ops.rope_qkv_cache(ops.gemv(x, w, bias), pos, cs, D, q2, k2, v2, slots, Hq, Hkv, D, k_scale=sc[0], v_scale=sc[1])
    for a, b in ((q1, q2), (kc, k2), (vc, v2)):
        assert torch.equal(a.float(), b.float())
