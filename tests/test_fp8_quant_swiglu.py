"""SiLU(gate) * up and its fp8 groups in one launch (``ome_fp8_quant_swiglu``)."""
import pytest
import torch

from ome_amd import ops


# one group, fewer and more pieces than threads, many rows
@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(1, 128), (3, 384), (700, 2048), (5, 2176), (0, 256)])
def test_same_bits_as_two_launches(M, K):
    torch.manual_seed(K)
    gu = (torch.randn(M, 2 * K, device="cuda") * 4).to(torch.bfloat16)
    if M:
        gu[0, :64] = -300   # exp overflows
        gu[-1, 0], gu[-1, K + 1] = float("inf"), float("nan")
        gu[M // 2, K:] = 0   # a group of zeros
    want_q, want_s = ops.fp8_quant(ops.act_and_mul(gu), 128) if M else (torch.empty(0, K, device="cuda"), torch.empty(0, K // 128, device="cuda"))
    q, s = ops._act_fp8_quant(gu, 0)
    assert q.shape == (M, K) and s.shape == (M, K // 128)
    assert torch.equal(q.view(torch.uint8), want_q.to(torch.float8_e4m3fn).view(torch.uint8))
    assert torch.equal(s.view(torch.int32), want_s.view(torch.int32))
