"""Causal prefill of four query heads to a kv head, 32 rows of two heads a wave (``csrc/kernels/prefill_pair.hip``)."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

# one and two tiles of 32 keys; rows and keys around a tile's edge, pairs of steps and one left over; more than the 32 tiles whose pages a
# wave looks up at a time; a workgroup an item, runs of pieces and (forced) equal pieces; more than 512 workgroups (fp8's rule), of more keys
# and of one page, one row and one key too; items of 11, 18 and 32 pieces, which are merged four at a time
SHAPES = [([1, 2, 32, 33], [1, 34, 32, 64], False), ([5, 31, 64, 97], [37, 95, 128, 1025], False), ([5, 31, 64, 97], [37, 95, 128, 1025], True),
          ([64], [2100], False), ([40, 3], [160, 2085], True), ([33] * 70, [33 + 31 * (i % 5) for i in range(70)], False),
          ([1, 2, 17, 33] * 28, [1, 34, 17, 65] * 28, False), ([40], [3000], False), ([100], [5000], False), ([64], [9000], False)]
P, D, HKV, DEV = 16, 128, 4, "cuda"


def _inputs(shape, cache, sinks):
    q_lens, kv_lens, force = SHAPES[shape]
    torch.manual_seed(shape)
    t = lambda a, c: torch.tensor(a, dtype=torch.int32, device=DEV).view(-1, c)  # noqa: E731
    pages = [-(-n // P) for n in kv_lens]
    kc = (torch.randn(sum(pages), HKV, P, D, device=DEV) * 0.5).to(cache)
    vc = (torch.randn(sum(pages), HKV, D, P, device=DEV) * 0.5).to(cache)
    perm = torch.randperm(sum(pages), device=DEV).int()
    bt = torch.zeros(len(pages), max(pages), dtype=torch.int32, device=DEV)
    for i, n in enumerate(pages):
        bt[i, :n] = perm[sum(pages[:i]):sum(pages[:i]) + n]
    cu = torch.tensor([sum(q_lens[:i]) for i in range(len(q_lens) + 1)], dtype=torch.int32, device=DEV)
    kl = torch.tensor(kv_lens, dtype=torch.int32, device=DEV)
    wide = torch.randn(sum(q_lens), 6 * HKV, D, device=DEV).to(torch.bfloat16)
    q = wide[:, :4 * HKV]   # rows apart, as in a fused projection
    items, split, comb, chunk, parts = ops.prefill_plan(q_lens, kv_lens, kv_heads=HKV, force=force)
    assert (parts > 0) == (force or max(kv_lens) > 2048) and (len(q_lens) < 9 or len(items) * HKV > 512)
    plan = ops.PrefillPlan(t(items, 2), t(split, 4), t(comb, 4), chunk, parts)
    return q, kc, vc, bt, cu, kl, plan, torch.randn(4 * HKV, device=DEV) if sinks else None


def _check(out, q, kc, vc, bt, cu, kl, scale, sinks):
    """A weight is rounded to bf16, of 8 bits, and so is the output: 2^-8 of the weighted sum of |v| and of the result at the most.  (A tile of 32 keys left out
    of 2100 changes some output by 0.010; the bound is some 0.003 there.)"""
    args = (bt, cu, kl, scale, -1, 0.5, 2.0, 0.0, sinks)
    want = ref.paged_prefill(q.float(), kc, vc, *args)
    size = ref.paged_prefill(q.float(), kc, vc.float().abs().to(vc.dtype), *args)
    assert bool(((out.float() - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5).all())


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2], ids=str)
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_matches_reference(shape, cache):
    q_lens, kv_lens, _ = SHAPES[shape]
    q, kc, vc, bt, cu, kl, plan, sinks = _inputs(shape, cache, shape % 2)
    out = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, k_scale=0.5, v_scale=2.0, sinks=sinks)
    _check(out, q, kc, vc, bt, cu, kl, 0.0884, sinks)
    # a NaN in the last key's V reaches items of 32 rows that see its tile of 32 keys at most
    rows = max(0, (kv_lens[-1] - 1) // 32 * 32 - (kv_lens[-1] - q_lens[-1])) // 32 * 32
    vc[bt[-1, -(-kv_lens[-1] // P) - 1].item(), :, :, (kv_lens[-1] - 1) % P] = float("nan")
    bad = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, k_scale=0.5, v_scale=2.0, sinks=sinks)
    first = sum(q_lens[:-1]) + rows
    assert torch.equal(bad[:first], out[:first]) and bool(bad[-1].isnan().all())


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn], ids=str)
@pytest.mark.parametrize("shape", [1, 2, 3, 5])
@pytest.mark.parametrize("scale", [-0.0884, 0.0])
def test_scales_that_turn_the_scores_round(shape, cache, scale):
    """The largest score is looked for before it is scaled, so these go to the general body."""
    q, kc, vc, bt, cu, kl, plan, sinks = _inputs(shape, cache, shape % 2)
    q = q * 100   # (scores of 25 and more either way: weights that were scaled by the wrong end of them would be infinite)
    out = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, scale, k_scale=0.5, v_scale=2.0, sinks=sinks)
    _check(out, q, kc, vc, bt, cu, kl, scale, sinks)
