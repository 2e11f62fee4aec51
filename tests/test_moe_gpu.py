"""MoE kernels on MI355X vs fp32 PyTorch references: routing, device align, grouped MFMA GEMM,
combine; plus a tiny-MoE engine with HIP-graph decode."""
import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (37, 8, 2), (256, 64, 8), (300, 128, 4), (5, 512, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_moe_route(T, E, k, dtype):
    logits = torch.randn(T, E, device=DEV, dtype=dtype)
    w, ids = ops.moe_route(logits, k, renorm=True)
    rw, rids = ref.moe_route(logits.float(), k, True)
    # the chosen experts' probabilities must equal the reference's top-k values (ties may reorder)
    assert torch.allclose(w, rw, atol=1e-5)
    p = torch.softmax(logits.float(), -1)
    got = torch.gather(p, 1, ids.long())
    assert torch.allclose(got / got.sum(-1, keepdim=True), w, atol=1e-5)
    assert (ids.sort(-1).values == rids.sort(-1).values).float().mean() > 0.99


@pytest.mark.parametrize("T,E,k,H,I", [(1, 8, 2, 256, 128), (64, 8, 2, 512, 256), (200, 16, 4, 256, 96),
                                       (7, 64, 6, 1024, 64), (513, 8, 2, 4096, 1024)])
@pytest.mark.parametrize("tile", ["64", "128"])
def test_fused_moe(T, E, k, H, I, tile, monkeypatch):
    monkeypatch.setenv("OME_MOE_TILE", tile)
    x = torch.randn(T, H, device=DEV, dtype=torch.bfloat16)
    w13 = torch.randn(E, 2 * I, H, device=DEV, dtype=torch.bfloat16) * 0.05
    w2 = torch.randn(E, H, I, device=DEV, dtype=torch.bfloat16) * 0.05
    logits = torch.randn(T, E, device=DEV)
    if T > 4:
        logits[:, -1] = -1e4  # an expert that receives no tokens
    tw, tid = ops.moe_route(logits, k, renorm=True)
    out = ops.fused_moe(x, tw, tid, w13, w2)
    want = ref.fused_moe(x, tw, tid, w13, w2)
    err = (out.float() - want.float()).abs().max().item()
    assert err < 3e-2 * max(1.0, want.float().abs().max().item()), err


def test_tiny_moe_engine_graphs():
    from ome_amd.runtime.engine import Engine, EngineArgs
    from ome_amd.runtime.request import SamplingParams

    g = Engine(EngineArgs(model="tiny-moe", device="cuda", max_running_requests=16, context_length=512))
    e = Engine(EngineArgs(model="tiny-moe", device="cuda", max_running_requests=16, context_length=512,
                          cuda_graph=False, overlap_schedule=False))
    prompts = [[3 + (i * 31 + j) % 1000 for j in range(10 + 7 * i)] for i in range(6)]
    sp = SamplingParams(max_new_tokens=16, ignore_eos=True)
    a = [r.output_ids for r in g.generate(prompts, sp)]
    b = [r.output_ids for r in e.generate(prompts, sp)]
    match = sum(x == y for x, y in zip(a, b))
    assert match >= 5, (a, b)  # bf16 batch-shape differences may flip a rare near-tie


@pytest.mark.parametrize("counts", [[1, 0, 255, 257, 0, 512, 3], [40] * 70, [0, 0, 700]], ids=lambda c: f"{len(c)}x{max(c)}")
@pytest.mark.parametrize("H,I", [(256, 128), (192, 224), (128, 1856)])
@pytest.mark.parametrize("kind", ["silu", "gelu", "bias", "relu2"])
def test_moe_prompt_tiles(monkeypatch, counts, H, I, kind):
    """256-row tiles: empty experts, tiles of one row and of all, more experts than lanes, widths that end inside a
    tile, every epilogue."""
    torch.manual_seed(H + I)
    E, n = len(counts), sum(counts)
    bf = lambda *s: torch.randn(*s, device=DEV).to(torch.bfloat16)  # noqa: E731
    gated = kind != "relu2"
    x, w13, w2 = bf(n, H + 8)[:, 8:], bf(E, 2 * I if gated else I, H) * 0.1, bf(E, H, I) * 0.1
    b13, b2 = (bf(E, 2 * I), bf(E, H)) if kind == "bias" else (None, None)
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])[torch.randperm(n)].to(DEV)[:, None]
    tw = torch.rand(n, 1, device=DEV)
    monkeypatch.setattr(ops, "MOE_PP_ROWS", 0)
    act = {"silu": 0, "gelu": 1, "bias": 0, "relu2": 4}[kind]
    got = ops.fused_moe(x, tw, ids.contiguous(), w13, w2, act, 1.0, b13, b2, gated).cpu().double()
    d = lambda t: t.cpu().double()  # noqa: E731
    want = torch.zeros(n, H, dtype=torch.float64)
    for e in range(E):
        r = (ids[:, 0] == e).nonzero()[:, 0].cpu()
        h = d(x)[r] @ d(w13[e]).T + (d(b13[e]) if b13 is not None else 0)
        if gated:
            g = h[:, :I]
            h = (torch.nn.functional.gelu(g, approximate="tanh") if kind == "gelu" else g * g.sigmoid()) * h[:, I:]
        else:
            h = h.clamp(min=0).square()
        want[r] = (h @ d(w2[e]).T + (d(b2[e]) if b2 is not None else 0)) * d(tw)[r]
    # bf16 roundings of the intermediate (two where the activation is a pass of its own), the expert's row and the output
    assert ((got - want).norm() / want.norm()).item() < 2.0 ** -7
    assert torch.isfinite(got).all()


@pytest.mark.parametrize("rows", [1, 64, 65, 128, 129, 192, 193, 256])
def test_moe_prompt_tile_quarters(monkeypatch, rows):
    """256-row tiles multiply the 64-row quarters that have rows: both sides of each quarter's edge, in an expert's only tile and
    in its second one, with one K step and with several."""
    for H, I in ((64, 64), (192, 224)):
        test_moe_prompt_tiles(monkeypatch, [rows, 256 + rows, 0, 3], H, I, "silu")


@pytest.mark.parametrize("counts", [[1, 0, 255, 257, 0, 512, 3], [40] * 70], ids=lambda c: f"{len(c)}x{max(c)}")
@pytest.mark.parametrize("H,I", [(256, 128), (192, 192), (128, 1856)])
@pytest.mark.parametrize("splits", [2, 3])
def test_moe_down_projection_in_pieces(monkeypatch, counts, H, I, splits):
    """Pieces of one K step, of unlike length, of many; the shared expert's rows on top."""
    splits = min(splits, I // 64)
    monkeypatch.setattr(ops, "moe_splits", lambda *a: splits)
    for kind in ("silu", "relu2"):
        test_moe_prompt_tiles(monkeypatch, counts, H, I, kind)
    torch.manual_seed(I)
    bf = lambda *s: torch.randn(*s, device=DEV).to(torch.bfloat16)  # noqa: E731
    x, w13, w2, add = bf(300, H), bf(4, 2 * I, H) * 0.1, bf(4, H, I) * 0.1, bf(300, H)
    tw, ids = torch.rand(300, 2, device=DEV), torch.rand(300, 4, device=DEV).topk(2).indices.int()
    got = ops.fused_moe(x, tw, ids, w13, w2, 0, 2.5, add=add.clone()).double()
    monkeypatch.setattr(ops, "moe_splits", lambda *a: 1)
    # without pieces each expert's row is rounded to bf16 before they are added, and the output either way
    plain = ops.fused_moe(x, tw, ids, w13, w2, 0, 2.5, add=add.clone()).double()
    assert ((got - plain).norm() / plain.norm()).item() < 2.0 ** -8


@pytest.mark.parametrize("tokens,splits", [(184, 2), (600, 2), (800, 1), (1500, 1), (1800, 2), (2600, 2), (3000, 1)])
def test_moe_pieces_where_they_are_faster(tokens, splits):
    assert ops.moe_splits(2 * tokens, 8, 4096, 14336) == splits


@pytest.mark.parametrize("E,k", [(1, 1), (64, 64), (65, 3), (200, 70), (512, 10)])
def test_moe_route_picks_in_order(E, k):
    """Ties go to the lower expert, zeros of both signs are ties, minus infinity comes last, NaN never (an expert
    id comes out all the same); also with more picks than lanes."""
    torch.manual_seed(E)
    logits = torch.randint(-3, 4, (9, E)).float()
    logits[1], logits[2], logits[3] = 0.0, -0.0, float("-inf")
    logits[2, ::2] = 0.0
    logits[4, E // 2:] = float("-inf")
    w, ids = (t.cpu() for t in ops.moe_route(logits.to(DEV), k, True, "sigmoid"))
    order = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :k]
    assert torch.equal(ids.long(), order)
    s = logits.double().sigmoid().gather(1, order)
    assert torch.allclose(w.double(), s / (s.sum(1, keepdim=True) + 1e-20), rtol=1e-5, atol=1e-7)
    nan = torch.full((2, E), float("nan"))
    nan[1, E // 2] = 1.0
    _, ids = ops.moe_route(nan.to(DEV), k, True, "sigmoid")
    assert ids[1, 0].item() == E // 2 and ((ids >= 0) & (ids < E)).all()


@pytest.mark.parametrize("E", [1, 64, 1023, 1024, 1025, 3000])
@pytest.mark.parametrize("n", [1, 5000])
def test_moe_align_offsets(E, n):
    torch.manual_seed(E + n)
    ids = torch.randint(0, E, (n,), dtype=torch.int32, device=DEV)
    off, srt, inv = (torch.full((s,), -1, dtype=torch.int32, device=DEV) for s in (E + 1, n, n))
    ops.call("ome_moe_align", ids.data_ptr(), n, E, off.data_ptr(), srt.data_ptr(), inv.data_ptr(), ops.stream_ptr())
    count = torch.bincount(ids.cpu().long(), minlength=E)
    assert torch.equal(off.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), count.cumsum(0)]))
    assert torch.equal(ids[srt.long()].cpu(), ids.cpu().sort().values)
    assert torch.equal(srt[inv.long()].cpu(), torch.arange(n, dtype=torch.int32))


@pytest.mark.parametrize("E", [1, 512])
@pytest.mark.parametrize("n", [3072, 3073, 8192, 8193, 32768, 32769])
def test_moe_align_of_many(E, n):
    """Assignments that threads keep, to the last of eight at a time and of 32 in all, and one more."""
    test_moe_align_offsets(E, n)


@pytest.mark.parametrize("E,e_tiles", [(1, 1), (64, 64), (300, 299), (1025, 1025)])
@pytest.mark.parametrize("n,bm", [(1, 64), (65, 64), (5000, 64), (5000, 128)])
def test_moe_align_tiles(E, e_tiles, n, bm):
    torch.manual_seed(E + n)
    ids = (torch.randint(0, E, (n,)) * torch.randint(0, 2, (n,))).to(torch.int32).to(DEV)   # half of them the first expert's
    s = ops._Sorted(ids, E, bm, e_tiles)
    off = torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(ids.cpu().long(), minlength=E).cumsum(0)]).tolist()
    want = [[e, m, off[e + 1], 0] for e in range(e_tiles) for m in range(off[e], off[e + 1], bm)]
    tiles = s.meta[:4 * s.max_tiles].view(-1, 4).tolist()
    assert tiles[:len(want)] == want and all(t[0] == -1 for t in tiles[len(want):]) and len(want) <= len(tiles)


@pytest.mark.parametrize("counts", [[1], [64, 0, 65], [0, 63, 128, 1, 0], [3] * 40, [0] * 30 + [130] * 12], ids=str)
@pytest.mark.parametrize("N,K", [(64, 64), (100, 128), (37, 192), (320, 320), (3000, 64)])
@pytest.mark.parametrize("gather", [True, False])
def test_streamed_experts_at_tile_edges(counts, N, K, gather):
    """Rows, weight rows and stages that fill no tile, experts without rows, few workgroups (four stages) and many (three)."""
    torch.manual_seed(N + K)
    E, n = len(counts), sum(counts)
    order = torch.randperm(n)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[order].to(torch.int32).to(DEV)
    x = torch.randn(n, K + 8, device=DEV).to(torch.bfloat16)[:, 8:] if gather else torch.randn(n, K, device=DEV).to(torch.bfloat16)
    w, b = (torch.randn(E, N, K, device=DEV) * K ** -0.5).to(torch.bfloat16), torch.randn(E, N, device=DEV).to(torch.bfloat16)
    s = ops._Sorted(ids, E, 64)
    assert ops.moe_tile_m(n, E, N) == 64
    got = ops._moe_gemm(x, s, s.ids if gather else None, 1 if gather else 0, w, n, b).cpu()
    rows = s.meta[-2 * n:-n].long().cpu() if gather else torch.arange(n)
    e = ids.cpu().long().sort().values
    want = torch.einsum("nk,nok->no", x.cpu().double()[rows], w.cpu().double()[e]) + b.cpu().double()[e]
    # fp32 sums of K products, one rounding to bf16: 2^-8 of each value (half a step), and 2^-24 K of the products' size
    assert torch.allclose(got.double(), want, rtol=2.0 ** -8, atol=2.0 ** -24 * K * 8)


@pytest.mark.parametrize("counts", [[1], [1] * 9, [2] * 13, [0, 63, 1, 0] + [0] * 3, [0] * 30 + [31] * 12 + [65], [5] * 40], ids=str)
@pytest.mark.parametrize("N,K", [(512, 64), (500, 128), (1024, 320), (24576, 64)])
def test_streamed_experts_in_runs(monkeypatch, counts, N, K):
    """An XCD's workgroups take a run of the tiles: as many tiles as there may be and fewer, fewer than XCDs, a multiple of 8 workgroups and not."""
    runs, call = [], ops.call
    monkeypatch.setattr(ops, "call", lambda fn, *a: (runs.append(a[-2]) if fn == "ome_moe_gemm_stream" else None, call(fn, *a)))
    test_streamed_experts_at_tile_edges(counts, N, K, True)
    assert runs == [1]


@pytest.mark.parametrize("counts,N,K", [([1, 0, 2, 1], 1024, 512), ([1, 1], 4096, 14336), ([1] * 6, 2688, 1856), ([0, 64, 3], 64, 128)], ids=str)
@pytest.mark.parametrize("gather", [True, False])
def test_streamed_experts_out_of_memory(counts, N, K, gather):
    """Few workgroups, four stages: rows and weights that no cache holds, so that each block is late and has to be waited for."""
    torch.manual_seed(N)
    E, n = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32).to(DEV)
    x, b = torch.randn(n, K, device=DEV).to(torch.bfloat16), torch.randn(E, N, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, N, K, device=DEV) * K ** -0.5).to(torch.bfloat16)
    s = ops._Sorted(ids, E, 64)
    assert ops.moe_tile_m(n, E, N) == 64 and -(-N // 64) * s.max_tiles <= 512
    rows = s.meta[-2 * n:-n].long() if gather else torch.arange(n, device=DEV)
    want = torch.cat([x[rows[ids == e]].double() @ w[e].double().t() + b[e].double() for e in range(E)])
    others = torch.empty(1 << 28, dtype=torch.float32, device=DEV)   # four times the last-level cache
    for i in range(4):
        others.fill_(i)
        got = ops._moe_gemm(x, s, s.ids if gather else None, 1 if gather else 0, w, n, b)
        # as above: 2^-8 of each value and 2^-24 K of the products' size
        assert torch.allclose(got.double(), want, rtol=2.0 ** -8, atol=2.0 ** -24 * K * 8)


@pytest.mark.parametrize("counts", [[1], [64, 0, 65], [0, 63, 128, 1, 0]], ids=str)
@pytest.mark.parametrize("N,K,shift", [(100, 96, 0), (37, 32, 4), (320, 224, 8), (100, 128, 4), (64, 192, 1)])
@pytest.mark.parametrize("gather", [True, False])
def test_experts_of_any_width_and_start(monkeypatch, counts, N, K, shift, gather):
    """64-row tiles where K is no multiple of 64 (the kernel that searches its tile itself), and where it is but rows start on no
    16-byte boundary (streamed, from a copy)."""
    torch.manual_seed(N + K)
    E, n = len(counts), sum(counts)
    order = torch.randperm(n)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[order].to(torch.int32).to(DEV)
    x = torch.randn(n, K + 8, device=DEV).to(torch.bfloat16)[:, shift:shift + K]
    w, b = (torch.randn(E, N, K, device=DEV) * K ** -0.5).to(torch.bfloat16), torch.randn(E, N, device=DEV).to(torch.bfloat16)
    s, ran, call = ops._Sorted(ids, E, 64), [], ops.call
    monkeypatch.setattr(ops, "call", lambda fn, *a: (ran.append(fn), call(fn, *a)))
    got = ops._moe_gemm(x, s, s.ids if gather else None, 1 if gather else 0, w, n, b).cpu()
    assert ran == ["ome_moe_gemm" if K % 64 else "ome_moe_gemm_stream"]
    rows = s.meta[-2 * n:-n].long().cpu() if gather else torch.arange(n)
    e = ids.cpu().long().sort().values
    want = torch.einsum("nk,nok->no", x.cpu().double()[rows], w.cpu().double()[e]) + b.cpu().double()[e]
    # fp32 sums of K products, one rounding to bf16: 2^-8 of each value (half a step), and 2^-24 K of the products' size
    assert torch.allclose(got.double(), want, rtol=2.0 ** -8, atol=2.0 ** -24 * K * 8)
