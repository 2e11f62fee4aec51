"""Merging the parts of paged decode attention (``paged_decode_reduce_kernel``)."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


# parts of 128 keys: two, around the 16 that are read at a time, around as many as a head has threads (64, 128), and one part beside them
@pytest.mark.parametrize("D,lens", [(128, [129, 2048, 2049, 60]), (128, [128 * 128, 128 * 128 + 1, 300, 33]), (64, [64 * 128 + 5, 200, 16 * 128, 1]),
                                    (256, [129, 17 * 128, 40, 1000])])
@pytest.mark.parametrize("dynamic", [False, True], ids=["spans", "own length"])
@pytest.mark.parametrize("sinks", [False, True], ids=["", "sinks"])
def test_parts(D, lens, dynamic, sinks):
    torch.manual_seed(D + len(lens))
    dev, P, Hq, Hkv, B = "cuda", 16, 8, 2, len(lens)
    pages = [-(-n // P) for n in lens]
    kc = torch.randn(sum(pages), Hkv, P, D, device=dev).to(torch.bfloat16)
    vc = torch.randn(sum(pages), Hkv, D, P, device=dev).to(torch.bfloat16)
    bt = torch.zeros(B, max(pages), dtype=torch.int32, device=dev)
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(sum(pages[:i]), sum(pages[:i]) + n, device=dev)
    q = torch.randn(B, Hq, D, device=dev).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32, device=dev)
    s = torch.randn(Hq, device=dev) if sinks else None
    ws = ops.DecodeWorkspace(B, Hq, D, max(lens), 0 if dynamic else 128, dev, parts=150 if dynamic else None)
    ws.part_o.fill_(float("nan"))   # parts that no key has are not read into a sum
    ws.part_ml.fill_(float("nan"))
    out = ops.paged_decode(q, kc, vc, bt, sl, D ** -0.5, ws, sinks=s)
    want = ref.paged_decode(q, kc, vc, bt, sl, D ** -0.5, sinks=s)
    # probabilities and output rounded to bf16 once each: 2^-9 of the largest |v| (about 5) apiece
    assert (out.float() - want.float()).abs().max().item() < 2 * 2.0 ** -9 * 5
