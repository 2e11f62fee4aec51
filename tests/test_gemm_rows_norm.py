"""One or two rows through a norm and the product after it in one launch (``ops.gemv_add``, ``ops.gemm_rows_norm``)."""
import pytest
import torch

from ome_amd import ops

pytestmark = pytest.mark.gpu


# K: one step of 64, fewer steps than stages, some pieces of a thread empty, all full; N: the fewest and more tiles than CUs
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("K,N", [(64, 24576), (192, 24576), (2112, 32768), (4096, 49152), (8192, 24576)])
def test_matches_norm_and_product(M, K, N):
    torch.manual_seed(K + M)
    dev, eps = "cuda", 1e-5
    res = torch.randn(M, K + 64, device=dev).to(torch.bfloat16)[:, :K]   # rows apart
    res[0] *= 30
    ln = (1 + 0.1 * torch.randn(K, device=dev)).to(torch.bfloat16)
    a = torch.randn(M, 512, device=dev).to(torch.bfloat16)
    wo = (torch.randn(K, 512, device=dev) * 0.05).to(torch.bfloat16)
    w = (torch.randn(N, K, device=dev) * K ** -0.5).to(torch.bfloat16)
    assert ops.gemm_rows_norm_ok(a, wo, res, ln, w)
    part, before = ops.gemv(a, wo), res.clone()
    ops.fused_add_rmsnorm(part, before, ln, eps)
    ops.gemv_add(a, wo, res)
    assert torch.equal(res, before)
    out = ops.gemm_rows_norm(res, ln, eps, w)
    r = res.double()
    x = (r * torch.rsqrt((r * r).mean(-1, keepdim=True) + eps) * ln.double()).to(torch.bfloat16).double()
    g, u = (x @ w.double().t()).view(M, N // 32, 2, 16).unbind(2)
    g, u = g.reshape(M, -1), u.reshape(M, -1)
    s = torch.nn.functional.silu(g)
    # the output's rounding, and 1 / rms of another order of sums: the rows round to the next bf16 here and there, one of them 2^-8 of its
    # product (silu' is below 1.1; fp32 sums are far below that)
    one = 2.0 ** -8 * x.abs().amax() * w.double().abs().amax()
    assert bool(((out.double() - s * u).abs() <= 2.0 ** -8 * (s * u).abs() + one * (1.1 * u.abs() + s.abs()) + one * one).all())
    assert torch.isnan(ops.gemm_rows_norm(torch.full_like(res, float("nan")), ln, eps, w)).all()


def test_takes_what_it_is_for():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")  # noqa: E731
    args = lambda M=1, K=1024, N=24576: [z(M, 512), z(K, 512), z(M, K), z(K), z(N, K)]  # noqa: E731
    assert ops.gemm_rows_norm_ok(*args())
    assert not ops.gemm_rows_norm_ok(*args(M=3)) and not ops.gemm_rows_norm_ok(*args(K=8256)) and not ops.gemm_rows_norm_ok(*args(N=16384))
    wide = args(K=4096)
    wide[0], wide[1] = z(1, 16384), z(4096, 16384)   # a projection that comes in pieces
    assert not ops.gemm_rows_norm_ok(*wide)
    odd = args()
    odd[3] = z(1025)[1:]
    assert not ops.gemm_rows_norm_ok(*odd)
    f32 = args()
    f32[2] = f32[2].float()
    assert not ops.gemm_rows_norm_ok(*f32)
