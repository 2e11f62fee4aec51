"""Merging the parts of paged decode attention (``paged_decode_reduce_kernel``)."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


PARTS = [(128, [129, 2048, 2049, 60]), (128, [128 * 128, 128 * 128 + 1, 300, 33]), (64, [64 * 128 + 5, 200, 16 * 128, 1]), (256, [129, 17 * 128, 40, 1000])]


# parts of 128 keys: two, around the 16 that are read at a time, around as many as a head has threads (64, 128), and one part beside them
@pytest.mark.parametrize("D,lens", PARTS)
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


@pytest.mark.parametrize("D,lens", PARTS + [(256, [257 * 128 + 3, 256 * 128])])
@pytest.mark.parametrize("dynamic", [False, True], ids=["spans", "own length"])
def test_every_part_counts(D, lens, dynamic):
    """Scores of zero, and values of a part in one dim (of its own among D parts) that make that dim of the output 1, or 1 + 2 where two parts share it:
    a part left out, or taken twice, changes it by a third and more.  Weights are exact, so values and output are rounded to bf16 alone."""
    dev, P, Hq, Hkv, B = "cuda", 16, 8, 2, len(lens)
    pages = [-(-n // P) for n in lens]
    kc = torch.zeros(sum(pages), Hkv, P, D, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros(sum(pages), Hkv, D, P, dtype=torch.bfloat16, device=dev)
    bt = torch.zeros(B, max(pages), dtype=torch.int32, device=dev)
    want = torch.zeros(B, 1, D, dtype=torch.float64)
    for i, n in enumerate(lens):
        at = sum(pages[:i])
        bt[i, :pages[i]] = torch.arange(at, at + pages[i], device=dev)
        for p in range(-(-n // 128)):
            keys = min(n, 128 * p + 128) - 128 * p
            value = torch.tensor(2.0 ** (p // D) * n / keys).to(torch.bfloat16)
            vc[at + 8 * p:at + min(8 * p + 8, pages[i]), :, p % D] = value.to(dev)
            want[i, 0, p % D] += value.double() * keys / n
    ws = ops.DecodeWorkspace(B, Hq, D, max(lens), 0 if dynamic else 128, dev, parts=260 if dynamic else None)
    ws.part_o.fill_(float("nan"))
    ws.part_ml.fill_(float("nan"))
    out = ops.paged_decode(torch.zeros(B, Hq, D, dtype=torch.bfloat16, device=dev), kc, vc, bt, torch.tensor(lens, dtype=torch.int32, device=dev), 0.1, ws)
    assert bool(((out.double().cpu() - want).abs() <= 2.0 ** -8 * want + 1e-6).all())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dynamic", [False, True], ids=["spans", "own length"])
@pytest.mark.parametrize("sinks", [False, True], ids=["", "sinks"])
def test_order_of_the_sum(D, dynamic, sinks):
    """Bit by bit: L = fma(l, 2^(m - M), L) and O = fma(l 2^(m - M), o, O) over a head's parts, one after the other, then the sink.  (Formed in 64 bits
    and rounded, which is the fma but for a double rounding of 2^-29 of the cases.  L as a sum of rounded products moved some outputs by a step of bf16.)"""
    torch.manual_seed(D + sinks)
    dev, P, Hq, Hkv, B = "cuda", 16, 8, 2, 64
    lens = [int(x) for x in torch.randint(129, 2500, (B,))]
    pages = -(-max(lens) // P)
    kc = torch.randn(pages, Hkv, P, D, device=dev).to(torch.bfloat16)
    vc = torch.randn(pages, Hkv, D, P, device=dev).to(torch.bfloat16)
    bt = torch.stack([torch.randperm(pages, dtype=torch.int32, device=dev) for _ in lens])
    s = torch.randn(Hq, device=dev) if sinks else None
    ws = ops.DecodeWorkspace(B, Hq, D, max(lens), 0 if dynamic else 128, dev, parts=12 if dynamic else None)
    out = ops.paged_decode(torch.randn(B, Hq, D, device=dev).to(torch.bfloat16), kc, vc, bt, torch.tensor(lens, dtype=torch.int32, device=dev),
                           D ** -0.5, ws, sinks=s).cpu()
    o = ws.part_o.view(B, Hq, ws.max_parts, D).cpu()
    ml = ws.part_ml.view(B, Hq, ws.max_parts, 2)

    def fma(a, b, c):
        return (a.double() * b.double() + c.double()).float()

    for b, n in enumerate(lens):
        span = max(128, -(-(-(-n // ws.max_parts)) // 128) * 128) if dynamic else 128
        parts = -(-n // span)
        m, l = ml[b, :, :parts, 0], ml[b, :, :parts, 1].cpu()
        M = m.max(1, keepdim=True).values
        e, M = torch.exp2(m - M).cpu(), M[:, 0].cpu()
        L, acc = torch.zeros(Hq), torch.zeros(Hq, D)
        for p in range(parts):
            L = fma(l[:, p], e[:, p], L)
            acc = fma((l[:, p] * e[:, p])[:, None], o[b, :, p], acc)
        if sinks:
            L = L + torch.exp2(fma(s.cpu(), torch.tensor(1.4426950408889634), -M).to(dev)).cpu()
        if parts > 1:
            assert torch.equal(out[b], (acc / L[:, None]).to(torch.bfloat16)), (b, n)
