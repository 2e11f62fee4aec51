"""Projections of up to 256 decode rows (csrc/kernels/gemm_rows.hip) against fp32 / fp64 products."""
import pytest
import torch

from ome_amd import ops
from ome_amd.models.quant import linear
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
D = "cuda"


def _operands(M, N, K, pad=0):
    g = torch.Generator(device=D).manual_seed(M * 7 + N + K)
    x = torch.empty(M + 3, K + pad, device=D, dtype=torch.bfloat16).normal_(generator=g)
    x[M:] = float("nan")   # past the last row: never read
    if pad:
        x[:, K:] = float("nan")
    w = torch.empty(N, K, device=D, dtype=torch.bfloat16).normal_(0, 0.05, generator=g)
    return x[:M, :K], w


# the edges of every row tile (32, 64, 128, 256), K from one step of 64 to uneven pieces, rows that lie apart
@pytest.mark.parametrize("M", [1, 5, 32, 33, 64, 65, 128, 129, 255, 256])
@pytest.mark.parametrize("N,K,pad", [(128, 64, 0), (384, 320, 8), (256, 2112, 0), (1024, 1024, 64)])
def test_product_and_pieces(M, N, K, pad):
    x, w = _operands(M, N, K, pad)
    exact = x.double() @ w.double().t()
    bias = torch.randn(N, device=D, dtype=torch.bfloat16)
    # bf16 rounds within 2^-9 of a value, K fp32 additions of random sign within about sqrt(K) 2^-24
    assert ops.gemm_rows_ok(x, w, bias)
    y = ops.gemm_rows(x, w, bias).double() - bias.double()
    assert (y - exact).abs().max() <= 2 ** -8 * (exact.abs() + bias.abs().double() + 1).max()
    assert (ops.gemm_rows(x, w).double() - exact).norm() <= 2 ** -8 * exact.norm()
    for splits in {1, min(3, K // 64), min(8, K // 64)}:
        part = ops.gemm_rows_parts(x, w, splits)
        assert part.shape == (splits, M, N)
        assert (part.double().sum(0) - exact).norm() <= 4e-6 * exact.norm()
    wide = torch.full((M, N + 12), 7.0, device=D, dtype=torch.bfloat16)
    ops.gemm_rows(x, w, out=wide[:, :N])
    assert torch.equal(wide[:, :N], ops.gemm_rows(x, w)) and (wide[:, N:] == 7.0).all()


@pytest.mark.parametrize("M", [5, 40, 100, 200, 256])
def test_silu_epilogue(M):
    x, w = _operands(M, 512, 640)
    il = ops.interleave_gate_up(w)
    g, u = (x.double() @ w.double().t()).chunk(2, -1)
    exact = torch.nn.functional.silu(g) * u
    assert (ops.gemm_rows(x, il, epi=2).double() - exact).norm() <= 2 ** -8 * exact.norm()


@pytest.mark.parametrize("M,H,splits", [(5, 128, 1), (64, 4096, 8), (256, 5120, 6), (33, 8192, 3), (7, 16384, 2)])
def test_norm_of_pieces(M, H, splits):
    part = torch.randn(splits, M, H, device=D)
    res = torch.randn(M, H, device=D, dtype=torch.bfloat16)
    w = torch.randn(H, device=D, dtype=torch.bfloat16)
    total = part.double().sum(0) + res.double()
    r0 = total.float().to(torch.bfloat16)
    y = ops.add_rmsnorm_parts(part, res, w, 1e-5)
    assert (res.double() - total).abs().max() <= 2 ** -8 * total.abs().max() and (res != r0).float().mean() < 1e-3
    assert (y.double() - ref.rmsnorm(res.float(), w.float(), 1e-5).double()).norm() <= 2 ** -8 * y.double().norm()


def test_rows_stay_apart():
    """A row that is not finite reaches no other; what the plan refuses stays refused."""
    x, w = _operands(70, 256, 512)
    clean = ops.gemm_rows(x, w)
    x = x.clone()
    x[13, 100], x[64, 3] = float("nan"), float("inf")
    y = ops.gemm_rows(x, w)
    keep = [i for i in range(70) if i not in (13, 64)]
    assert torch.equal(y[keep], clean[keep]) and y[13].isnan().all() and not y[64].isfinite().any()
    w = torch.zeros(24576, 128, device=D, dtype=torch.bfloat16)
    x = torch.zeros(300, 132, device=D, dtype=torch.bfloat16)
    assert ops.gemm_rows_plan(x[:9, :128].contiguous(), w)
    for bad in (x[:257, :128], x[:9, :128], x[:9, 1:129], x[:0, :128], x[:9, :128].float(), x[:9, :128].contiguous().t()):
        assert not ops.gemm_rows_plan(bad, w)   # too many rows, rows or start unaligned, none, another type, columns apart
    assert not ops.gemm_rows_plan(x[:9, :128].contiguous(), w[:24576 - 64])
    assert not ops.gemm_rows_plan(x[:9, :128].contiguous(), w[:36864 - 24576])


def test_replayed_in_a_graph():
    x, w = _operands(48, 1024, 1024)
    res0, nw = torch.randn(48, 1024, device=D, dtype=torch.bfloat16), torch.ones(1024, device=D, dtype=torch.bfloat16)
    res = res0.clone()
    want = ops.add_rmsnorm_parts(ops.gemm_rows_parts(x, w, 4), res, nw, 1e-5)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        got = ops.add_rmsnorm_parts(ops.gemm_rows_parts(x, w, 4), res, nw, 1e-5)
    for _ in range(3):
        res.copy_(res0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        torch.randn(1 << 20, device=D)


def test_linear_refuses_and_broadcasts_as_the_library():
    """Widths, biases and outputs of other sizes, operands of other devices and gradients, at a size that the kernel takes."""
    g = torch.Generator(device=D).manual_seed(1)
    x, w, b = (torch.empty(*s, device=D, dtype=torch.bfloat16).normal_(generator=g) for s in ((9, 128), (24576, 128), (24576,)))
    assert ops.gemm_rows_plan(x, w, b)
    for args in ((x[:, :64].contiguous(), w), (x, w, b[:128].contiguous()), (x, w, b.cpu()), (x, w.cpu())):
        with pytest.raises(RuntimeError):
            linear(*args)
    want = torch.nn.functional.linear(x, w, b[:1])
    assert torch.equal(linear(x, w, b[:1]), want)
    y, wanted = (t.clone().requires_grad_() for t in (x, x))
    linear(y, w, b).float().square().sum().backward()
    torch.nn.functional.linear(wanted, w, b).float().square().sum().backward()
    assert torch.equal(y.grad, wanted.grad)
