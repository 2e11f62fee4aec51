"""Kernels of the recurrent layers at the sizes where their tiles end, on gfx950: the short convolution (tiles
of 16 rows), the gated norm with 16-byte pieces, and the chunked scans (chunks of 32 rows)."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16

# tile and chunk edges, empty sequences, rows shorter than the taps; 70: more than one wave of sequences
LENS = [[1, 0, 2, 3], [2, 0, 1], [15, 16, 17], [31, 0, 32, 33, 1], [64, 65], [97], [1, 40] + [1] * 68]


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def seqs(lens, slots):
    """(cu, slot, reset) with scattered slots; every third sequence starts here."""
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return i32(cu), i32([(5 * s + 3) % slots for s in range(len(lens))]), i32([int(s % 3 == 1) for s in range(len(lens))])


def cpu(*t):
    return [x.cpu() if x is not None else None for x in t]


@pytest.mark.parametrize("lens", LENS, ids=str)
@pytest.mark.parametrize("K,C,off", [(4, 1032, 8), (4, 37, 1), (2, 64, 0), (3, 520, 8), (5, 72, 8), (6, 16, 0)])
def test_short_conv(lens, K, C, off):
    torch.manual_seed(K)
    T, slots = sum(lens), 71
    x = torch.randn(T, C + off, device=DEV).to(BF)[:, off:]
    w, b = torch.randn(C, K, device=DEV).to(BF), torch.randn(C, device=DEV).to(BF) if K != 3 else None
    st = torch.randn(slots, C, K - 1, device=DEV).to(BF)
    sr, sq = st.cpu(), seqs(lens, slots)
    want = ref.ssm_conv1d(*cpu(x, w, b), sr, *cpu(*sq), torch.empty(T, C, dtype=BF))
    got = ops.ssm_conv1d(x, w, b, st, *sq)
    # one bf16 rounding of a sum of K + 1 fp32 products (K + 2 roundings of at most its largest partial sum)
    assert torch.allclose(got.cpu().float(), want.float(), rtol=2.0 ** -7, atol=1e-5)
    assert torch.equal(st.cpu(), sr)


def test_short_conv_in_place():
    """The output may be the input."""
    torch.manual_seed(1)
    sq, C = seqs([40, 1, 19], 4), 256
    x, w, st = torch.randn(60, C, device=DEV).to(BF), torch.randn(C, 4, device=DEV).to(BF), torch.randn(4, C, 3, device=DEV).to(BF)
    s2 = st.clone()
    want = ops.ssm_conv1d(x, w, None, st, *sq)
    got = ops.ssm_conv1d(x, w, None, s2, *sq, out=x)
    assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=1e-5) and torch.equal(st, s2)


@pytest.mark.parametrize("group", [64, 128, 256, 512, 1024, 2048])
@pytest.mark.parametrize("mode", [(False, False, "silu"), (True, False, "silu"), (False, True, "silu"), (True, True, "silu"),
                                  (True, True, "sigmoid")])
@pytest.mark.parametrize("rows,off", [(1, 8), (37, 8), (9, 1)])
def test_gated_norm(group, mode, rows, off):
    torch.manual_seed(group)
    first, exact, gate = mode
    y = torch.randn(rows, 3 * group + off, device=DEV).to(BF)[:, off:]   # off 1: rows that 16-byte loads cannot take
    z = torch.randn(rows, 3 * group + 16, device=DEV).to(BF)[:, 16:]
    w = (1 + 0.2 * torch.randn(group if first else 3 * group, device=DEV)).to(BF)
    want = ref.gated_rmsnorm(*cpu(y, z, w), group, 1e-5, first, exact, gate).float()
    got = ops.gated_rmsnorm(y, z, w, group, 1e-5, first, exact, gate).cpu().float()
    # up to three bf16 roundings, each of which a last-bit difference of the fp32 norm can turn by one step
    assert torch.allclose(got, want, rtol=2.0 ** -6, atol=1e-6)
