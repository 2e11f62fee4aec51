"""Long-range prefill attention dealt out as equal runs of 64-key stages (``ops._prefill_runs``)."""
import random

import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref


def _spans(split, nb, ends):
    """{item: [(first key, past the last, part)]} of a plan's pieces, as the kernel reads them, and each run's stages."""
    pieces, spans, load = split[:-nb], {}, []
    for i, (s, r, c, part) in enumerate(pieces):
        nxt = pieces[i + 1] if i + 1 < len(pieces) and part >= 0 else None
        hi = nxt[2] if nxt and nxt[:2] == (s, r) else ends[s, r]
        spans.setdefault((s, r), []).append((c, hi, part))
        load.append(-(-(hi - c) // 64))
    return spans, [sum(load[a:b]) for a, b, _, _ in split[-nb:]]


@pytest.mark.parametrize("seed", range(40))
def test_runs_cover_every_item_once(seed):
    rng = random.Random(seed)
    n = rng.randint(1, 6)
    q = [rng.choice([1, 31, 32, 33, rng.randint(1, 3000)]) for _ in range(n)]
    kv = [a + rng.choice([0, 5, rng.randint(2000, 20000)]) for a in q]
    heads = rng.choice([1, 2, 4, 8, 16, 32])
    items, split, comb, chunk, parts = ops.prefill_plan(q, kv, kv_heads=heads)
    if chunk >= 0:
        return
    ends = {(s, r): kv[s] - q[s] + min(r + 32, q[s]) for s, r in items}
    spans, load = _spans(split, -chunk, ends)
    runs = split[chunk:]
    assert -chunk * heads <= 512 and runs[0][0] == 0 and runs[-1][1] == len(split) + chunk
    assert all(a[0] < a[1] for a in runs) and all(a[1] == b[0] for a, b in zip(runs, runs[1:]))
    assert list(spans) == [tuple(i) for i in items]
    for item, v in spans.items():
        assert v[0][0] == 0 and v[-1][1] == ends[item] and all(a[1] == b[0] and a[1] % 64 == 0 for a, b in zip(v, v[1:]))
        assert all(lo < hi for lo, hi, _ in v) and (v[0][2] < 0) == (len(v) == 1)
    cut = [v for v in spans.values() if len(v) > 1]
    assert [p for v in cut for *_, p in v] == list(range(parts))
    assert [(i, v[0][2], len(v)) for i, v in spans.items() if len(v) > 1] == [((s, r), p, m) for s, r, p, m in comb]
    assert max(load) <= sum(load) / len(load) + 8


@pytest.mark.gpu
@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv", [([64], [2100], 32, 8), ([33, 1, 90], [4097, 2200, 90], 4, 1),
                                                   ([700], [2749], 16, 4)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn], ids=str)
@pytest.mark.parametrize("mode", ["plain", "softcap", "window", "sinks"])
def test_runs_match_reference(q_lens, kv_lens, Hq, Hkv, cache, mode):
    torch.manual_seed(sum(kv_lens))
    D, P, dev = 128, 16, "cuda"
    t = lambda a, c: torch.tensor(a, dtype=torch.int32, device=dev).view(-1, c)  # noqa: E731
    pages = [-(-n // P) for n in kv_lens]
    kc = (torch.randn(sum(pages) + 1, Hkv, P, D, device=dev) * 0.5).to(cache)
    vc = (torch.randn(sum(pages) + 1, Hkv, D, P, device=dev) * 0.5).to(cache)
    perm = (torch.randperm(sum(pages), device=dev) + 1).int()
    bt = torch.zeros(len(pages), max(pages), dtype=torch.int32, device=dev)
    for i, n in enumerate(pages):
        bt[i, :n] = perm[sum(pages[:i]):sum(pages[:i]) + n]
    cu = torch.tensor([sum(q_lens[:i]) for i in range(len(q_lens) + 1)], dtype=torch.int32, device=dev)
    kl = torch.tensor(kv_lens, dtype=torch.int32, device=dev)
    q = torch.randn(sum(q_lens), Hq, D, device=dev).to(torch.bfloat16)
    items, split, comb, chunk, parts = ops.prefill_plan(q_lens, kv_lens, kv_heads=Hkv)
    assert chunk < 0 and parts > 0
    plan = ops.PrefillPlan(t(items, 2), t(split, 4), t(comb, 4), chunk, parts)
    kw = {"softcap": dict(softcap=20.0), "window": dict(window=300), "sinks": dict(sinks=torch.randn(Hq, device=dev))}.get(mode, {})
    out = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, **kw)
    want = ref.paged_prefill(q, kc, vc, bt, cu, kl, 0.0884, kw.get("window", -1), 1.0, 1.0, kw.get("softcap", 0.0),
                             kw.get("sinks"))
    # probabilities and output rounded to bf16 once each: 2^-9 of the largest |v| (about 2.3) apiece
    assert (out.float() - want.float()).abs().max().item() < 2 * 2.0 ** -9 * 2.5


@pytest.mark.gpu
@pytest.mark.parametrize("q_lens,kv_lens,Hq,Hkv", [([28, 28], [1899, 1899], 32, 8), ([139], [1539], 32, 8), ([1], [1089], 4, 1), ([33, 2], [1120, 2048], 16, 4)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn], ids=str)
def test_runs_of_shorter_contexts_match_reference(q_lens, kv_lens, Hq, Hkv, cache):
    test_runs_match_reference(q_lens, kv_lens, Hq, Hkv, cache, "plain")


@pytest.mark.parametrize("q,kv,runs", [([40], [1088], False), ([40], [1089], True), ([28, 28], [1899, 1899], True), ([300], [1300], True),
                                       ([1900], [1900], False), ([200] * 4, [1700] * 4, False), ([2000], [4000], False), ([3000], [5000], False)])
def test_runs_where_they_are_faster(q, kv, runs):
    assert (ops.prefill_plan(q, kv)[3] < 0) == runs


@pytest.mark.parametrize("q,kv", [([64], [15936]), ([256], [4096]), ([33, 64], [9000, 3000]), ([512], [8192]), ([1500], [7600])])
def test_plan_of_other_layers_is_in_equal_chunks(q, kv):
    """Layers with a window, soft-capping or ALiBi: chunks where the items are too few, none where they fill the chip."""
    assert ops.prefill_plan(q, kv)[3] < 0
    items, split, comb, chunk, parts = ops.prefill_plan(q, kv, runs=False)
    if len(items) * 8 >= 256:
        assert chunk == parts == 0 and not split
    else:
        assert chunk >= 128 and chunk % 64 == 0 and len(split) >= 32 and parts > 0


@pytest.mark.parametrize("model,change,other", [("tiny-llama", {}, False), ("tiny-llama", {"sliding_window": 512}, True),
                                                ("tiny-gemma2", {}, True)])
def test_runner_sends_the_other_plan(monkeypatch, model, change, other):
    """... along with the runs, for a model that has such layers."""
    import dataclasses

    from ome_amd.models.config import preset
    from ome_amd.runtime.model_runner import ModelRunner
    from ome_amd.runtime.request import Request, SamplingParams
    from ome_amd.runtime.scheduler import ScheduledChunk, StepBatch

    cfg = dataclasses.replace(preset(model), max_position_embeddings=4096, **change)
    runner = ModelRunner(cfg, device="cpu", dtype=torch.float32, max_running=2, max_context=4096, max_total_tokens=8192, cuda_graph=False)
    seen = []
    forward = runner.model.forward
    monkeypatch.setattr(runner.model, "forward", lambda ids, meta, *a: (seen.append(meta.items), forward(ids, meta, *a))[1])
    r = Request([3] * 3064, SamplingParams(ignore_eos=True))
    r.pages, r.req_slot, r.num_cached = list(range(1, 193)), runner.slots.alloc(), 3000
    runner.slots.set_pages(r.req_slot, 0, r.pages)
    runner.slots.flush()
    runner.launch(StepBatch("prefill", [ScheduledChunk(r, 3000, 64, True)]))
    plan = seen[0]
    assert plan.chunk < 0 and len(plan.split) + plan.chunk > 2
    assert (plan.other.chunk >= 128 and len(plan.other.split) == plan.other.parts > 2) if other else not plan.other.parts


@pytest.mark.gpu
@pytest.mark.parametrize("kw,other,chunked", [(dict(window=900), True, True), (dict(softcap=20.0), True, True), (dict(window=-1024), True, True),
                                              ({}, True, False), (dict(window=900), False, False), (dict(window=300), True, None)], ids=str)
def test_other_layers_run_their_plan(monkeypatch, kw, other, chunked):
    """A window over a long range with few rows is split into chunks, as is all that the kernel's fast body does not
    take; the runs serve a caller that has no other plan."""
    torch.manual_seed(3)
    Hq, Hkv, D, P, n, q_len, dev = 8, 2, 128, 16, 3000, 40, "cuda"
    t = lambda a, c: torch.tensor(a, dtype=torch.int32, device=dev).view(-1, c)  # noqa: E731
    pages = -(-n // P)
    kc, vc = torch.randn(pages + 1, Hkv, P, D, device=dev).bfloat16(), torch.randn(pages + 1, Hkv, D, P, device=dev).bfloat16()
    bt = (torch.randperm(pages, device=dev) + 1).int().view(1, -1)
    cu, kl = torch.tensor([0, q_len], dtype=torch.int32, device=dev), torch.tensor([n], dtype=torch.int32, device=dev)
    q = torch.randn(q_len, Hq, D, device=dev).bfloat16()
    items, split, comb, chunk, parts = ops.prefill_plan([q_len], [n], kv_heads=Hkv)
    _, split2, comb2, chunk2, parts2 = ops.prefill_plan([q_len], [n], kv_heads=Hkv, runs=False)
    plan = ops.PrefillPlan(t(items, 2), t(split, 4), t(comb, 4), chunk, parts,
                           other=ops.PrefillPlan(t(items, 2), t(split2, 4), t(comb2, 4), chunk2, parts2) if other else None)
    calls = []
    call = ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (calls.append((name, a)), call(name, *a))[1])
    out = ops.paged_prefill(q, kc, vc, bt, cu, kl, plan, 0.0884, **kw)
    (name, a), = [c for c in calls if c[0].startswith("ome_paged_prefill")]
    if chunked is None:   # a narrow window: its items as they are
        assert name == "ome_paged_prefill"
    else:
        assert name == "ome_paged_prefill_split" and (a[10] == 0) == chunked and (a[13] == (chunk2 if chunked else 0))
    want = ref.paged_prefill(q, kc, vc, bt, cu, kl, 0.0884, kw.get("window", -1), 1.0, 1.0, kw.get("softcap", 0.0), None)
    # probabilities and output rounded to bf16 once each: 2^-9 of the largest |v| (about 4.5) apiece
    assert (out.float() - want.float()).abs().max().item() < 2 * 2.0 ** -9 * 5
