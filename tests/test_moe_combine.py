"""Weighted sum of a token's experts (``moe_combine_kernel``)."""
import pytest
import torch

from ome_amd import ops


# experts: every way that they come in batches of 8, 4, 2 and 1; columns: one piece, a workgroup's, and more than a workgroup's
@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 2, 3, 4, 6, 7, 8, 10, 15, 17])
@pytest.mark.parametrize("T,H", [(1, 8), (5, 2048), (3, 2056)])
@pytest.mark.parametrize("with_add", [False, True])
def test_sum(k, T, H, with_add):
    torch.manual_seed(k * H)
    y = torch.randn(T * k, H, device="cuda").to(torch.bfloat16)
    w = torch.rand(T, k, device="cuda")
    inv = torch.randperm(T * k, device="cuda").int()
    add = torch.randn(T, H, device="cuda").to(torch.bfloat16) if with_add else None
    terms = w.double()[..., None] * y.double()[inv.long()].view(T, k, H)
    want = 2.5 * terms.sum(1) + (0 if add is None else add.double())
    out = ops._combine(y, w, inv, T, k, H, 2.5, add)
    assert with_add == (out is add)
    # one rounding to bf16, whose 8 bits make half a last place up to 2^-8 of the value, and the sum in fp32
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.5 * (k + 2) * 2.0 ** -24 * terms.abs().sum(1) * 2 + 1e-30).all())
