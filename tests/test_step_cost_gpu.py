"""The step-cost table times the kernels that a step's forward runs."""
import dataclasses

import pytest
import torch

from ome_amd import ops
from ome_amd.models import quant
from ome_amd.models.config import preset
from ome_amd.runtime.model_runner import ModelRunner
from ome_amd.runtime.request import Request, SamplingParams
from ome_amd.runtime.scheduler import ScheduledChunk, StepBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cache", ["auto", "fp8"])
def test_probe_runs_the_forwards_kernels(cache, monkeypatch):
    """Two layers of an 8B model: the same projections and norms, by the same kernels and plans, at row counts on both sides of every
    kernel's range."""
    cfg = dataclasses.replace(preset("llama-3-8b"), num_layers=2, vocab_size=1024)
    r = ModelRunner(cfg, device="cuda", max_running=4, max_context=1024, max_total_tokens=4096, cuda_graph=False, kv_cache_dtype_name=cache)
    seen, probed = [], {}
    call, library, probe = ops.call, torch.nn.functional.linear, r.model.gemm_probe

    def record(fn, *args, **kw):
        if fn in ("ome_gemm_rows", "ome_gemm_sk", "ome_add_rmsnorm_parts", "ome_fused_add_rmsnorm"):
            seen.append((fn, *(a for a in args if isinstance(a, (int, float)) and abs(a) < 1 << 20)))   # sizes, strides and plans; no addresses
        return call(fn, *args, **kw)

    def record_library(x, w, b=None):
        seen.append(("library", *x.shape, *w.shape))
        return library(x, w, b)

    def record_probe(i, x, *args):
        seen.clear()
        probe(i, x, *args)
        probed[x.shape[0]] = list(seen)

    monkeypatch.setattr(ops, "call", record)
    monkeypatch.setattr(quant.F, "linear", record_library)
    monkeypatch.setattr(r.model, "gemm_probe", record_probe)
    assert r.measure_step_cost(320, grid=64, reps=1) is not None
    for M in (64, 256, 320):
        q = Request(list(range(3, 3 + M)), SamplingParams(ignore_eos=True))
        q.pages, q.req_slot = list(range(1, 1 + -(-M // 16))), r.slots.alloc()
        r.slots.set_pages(q.req_slot, 0, q.pages)
        r.slots.flush()
        seen.clear()
        r.launch(StepBatch("prefill", [ScheduledChunk(q, 0, M, True)]))
        torch.cuda.synchronize()
        r.slots.free(q.req_slot)
        one = len(probed[M])
        assert seen[:2 * one] == 2 * probed[M], M
        assert any(s[0] == "ome_add_rmsnorm_parts" for s in probed[M]) == (cache == "auto" and M <= 256)
