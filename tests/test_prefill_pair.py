"""Causal prefill of four query heads to a kv head, 32 rows of two heads a wave (``csrc/kernels/prefill_pair.hip``)."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

# one and two tiles of 32 keys; rows and keys around a tile's edge, pairs of steps and one left over; more than the 32 tiles whose pages a
# wave looks up at a time; a workgroup an item, runs of pieces and (forced) equal pieces; more than 512 workgroups (fp8's rule)
SHAPES = [([1, 2, 32, 33], [1, 34, 32, 64], False), ([5, 31, 64, 97], [37, 95, 128, 1025], False), ([5, 31, 64, 97], [37, 95, 128, 1025], True),
          ([64], [2100], False), ([40, 3], [160, 2085], True), ([33] * 70, [33 + 31 * (i % 5) for i in range(70)], False)]


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2], ids=str)
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_matches_reference(shape, cache):
    q_lens, kv_lens, force = SHAPES[shape]
    torch.manual_seed(shape)
    D, P, Hkv, dev = 128, 16, 4, "cuda"
    t = lambda a, c: torch.tensor(a, dtype=torch.int32, device=dev).view(-1, c)  # noqa: E731
    pages = [-(-n // P) for n in kv_lens]
    kc = (torch.randn(sum(pages), Hkv, P, D, device=dev) * 0.5).to(cache)
    vc = (torch.randn(sum(pages), Hkv, D, P, device=dev) * 0.5).to(cache)
    perm = torch.randperm(sum(pages), device=dev).int()
    bt = torch.zeros(len(pages), max(pages), dtype=torch.int32, device=dev)
    for i, n in enumerate(pages):
        bt[i, :n] = perm[sum(pages[:i]):sum(pages[:i]) + n]
    cu = torch.tensor([sum(q_lens[:i]) for i in range(len(q_lens) + 1)], dtype=torch.int32, device=dev)
    kl = torch.tensor(kv_lens, dtype=torch.int32, device=dev)
    wide = torch.randn(sum(q_lens), 6 * Hkv, D, device=dev).to(torch.bfloat16)
    q = wide[:, :4 * Hkv]   # rows apart, as in a fused projection
    items, split, comb, chunk, parts = ops.prefill_plan(q_lens, kv_lens, kv_heads=Hkv, force=force)
    assert (parts > 0) == (force or max(kv_lens) > 2048)
    plan = ops.PrefillPlan(t(items, 2), t(split, 4), t(comb, 4), chunk, parts)
    sinks = torch.randn(4 * Hkv, device=dev) if shape % 2 else None
    out = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, k_scale=0.5, v_scale=2.0, sinks=sinks)
    want = ref.paged_prefill(q, kc, vc, bt, cu, kl, 0.0884, -1, 0.5, 2.0, 0.0, sinks)
    # probabilities and output rounded to bf16 once each: 2^-9 of the largest |v| (with its scale 2 * 2.7) apiece
    assert (out.float() - want.float()).abs().max().item() < 2 * 2.0 ** -9 * 5.4
    # a NaN in the last key's V reaches items of 32 rows that see its tile of 32 keys at most
    rows = max(0, (kv_lens[-1] - 1) // 32 * 32 - (kv_lens[-1] - q_lens[-1])) // 32 * 32
    vc[bt[-1, pages[-1] - 1].item(), :, :, (kv_lens[-1] - 1) % P] = float("nan")
    bad = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, k_scale=0.5, v_scale=2.0, sinks=sinks)
    first = sum(q_lens[:-1]) + rows
    assert torch.equal(bad[:first], out[:first]) and bool(bad[-1].isnan().all())
