"""One or two rows through a norm and the product after it in one launch (``ops.gemv_add``, ``ops.gemm_rows_norm``)."""
import dataclasses

import pytest
import torch

from ome_amd import ops
from ome_amd.models.config import preset
from ome_amd.runtime.model_runner import ModelRunner
from ome_amd.runtime.request import Request, SamplingParams
from ome_amd.runtime.scheduler import ScheduledChunk, StepBatch

pytestmark = pytest.mark.gpu


# K: one step of 64, fewer steps than stages, some pieces of a thread empty, all full; N: the fewest and more tiles than CUs
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("K,N", [(64, 24576), (192, 24576), (2112, 32768), (4096, 49152), (8192, 24576)])
def test_matches_norm_and_product(M, K, N):
    torch.manual_seed(K + M)
    dev, eps = "cuda", 1e-5
    res = torch.randn(M, K + 64, device=dev).to(torch.bfloat16)[:, :K]   # rows apart
    res[0] *= 30
    ln = (1 + 0.1 * torch.randn(K, device=dev)).to(torch.bfloat16)
    a = torch.randn(M, 512, device=dev).to(torch.bfloat16)
    wo = (torch.randn(K, 512, device=dev) * 0.05).to(torch.bfloat16)
    w = (torch.randn(N, K, device=dev) * K ** -0.5).to(torch.bfloat16)
    assert ops.gemm_rows_norm_ok(a, wo, res, ln, w)
    part, before = ops.gemv(a, wo), res.clone()
    ops.fused_add_rmsnorm(part, before, ln, eps)
    ops.gemv_add(a, wo, res)
    assert torch.equal(res, before)
    out = ops.gemm_rows_norm(res, ln, eps, w)
    assert torch.equal(out, ops.gemm_rows(part, w, epi=2))   # (the norm's sums in the same order, the products too)
    r = res.double()
    x = (r * torch.rsqrt((r * r).mean(-1, keepdim=True) + eps) * ln.double()).to(torch.bfloat16).double()
    g, u = (x @ w.double().t()).view(M, N // 32, 2, 16).unbind(2)
    g, u = g.reshape(M, -1), u.reshape(M, -1)
    s = torch.nn.functional.silu(g)
    # the output's rounding, and 1 / rms of another order of sums: the rows round to the next bf16 here and there, one of them 2^-8 of its
    # product (silu' is below 1.1; fp32 sums are far below that)
    one = 2.0 ** -8 * x.abs().amax() * w.double().abs().amax()
    assert bool(((out.double() - s * u).abs() <= 2.0 ** -8 * (s * u).abs() + one * (1.1 * u.abs() + s.abs()) + one * one).all())
    assert torch.isnan(ops.gemm_rows_norm(torch.full_like(res, float("nan")), ln, eps, w)).all()


def test_takes_what_it_is_for():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")  # noqa: E731
    args = lambda M=1, K=1024, N=24576: [z(M, 512), z(K, 512), z(M, K), z(K), z(N, K)]  # noqa: E731
    assert ops.gemm_rows_norm_ok(*args())
    assert not ops.gemm_rows_norm_ok(*args(M=3)) and not ops.gemm_rows_norm_ok(*args(K=8256)) and not ops.gemm_rows_norm_ok(*args(N=16384))
    wide = args(K=4096)
    wide[0], wide[1] = z(1, 16384), z(4096, 16384)   # a projection that comes in pieces
    assert not ops.gemm_rows_norm_ok(*wide)
    odd = args()
    odd[3] = z(1025)[1:]
    assert not ops.gemm_rows_norm_ok(*odd)
    f32 = args()
    f32[2] = f32[2].float()
    assert not ops.gemm_rows_norm_ok(*f32)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("mode", ["decode", "prefill"])
def test_a_model_takes_it(rows, mode, monkeypatch):
    """Two layers of an 8B model: steps of one and two rows give the same bits with the norm as a launch of its own."""
    cfg = dataclasses.replace(preset("llama-3-8b"), num_layers=2, vocab_size=1024)
    r = ModelRunner(cfg, device="cuda", max_running=4, max_context=1024, max_total_tokens=4096, cuda_graph=False, keep_logits=True)
    took, norm = [], ops.gemm_rows_norm
    monkeypatch.setattr(ops, "gemm_rows_norm", lambda *a: (took.append(a[0].shape[0]), norm(*a))[1])
    reqs = []
    for i in range(rows if mode == "decode" else 1):
        reqs.append(Request([5 + i, 7, 9], SamplingParams(ignore_eos=True)))
        reqs[i].pages, reqs[i].req_slot = [1 + i], r.slots.alloc()
        r.slots.set_pages(reqs[i].req_slot, 0, reqs[i].pages)
    r.slots.flush()
    before = 0
    if mode == "decode":
        before = 2
        r.launch(StepBatch("prefill", [ScheduledChunk(q, 0, 2, True, want=[1]) for q in reqs]))
        for q in reqs:
            q.num_cached = 2
    took.clear()
    step = lambda: r.launch(StepBatch(mode, [ScheduledChunk(q, before, 1 if mode == "decode" else rows, True, want=[0]) for q in reqs])).logits.clone()  # noqa: E731
    folded = step()
    assert took == 2 * [rows]
    monkeypatch.setattr(ops, "gemm_rows_norm_ok", lambda *a: False)
    assert torch.equal(folded, step()) and took == 2 * [rows]
