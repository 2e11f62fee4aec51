"""MLA attention kernel (csrc/kernels/mla.hip), grouped routing, and the DeepSeek model on the GPU."""
import random

import pytest
import torch

from ome_amd import ops
from ome_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _setup(lens, seed=0, dk=576):
    g = torch.Generator().manual_seed(seed)
    pages_per_row = -(-max(lens) // 16) + 1
    num_pages = len(lens) * pages_per_row + 1
    cache = (torch.randn(num_pages, 16, dk, generator=g) * 0.5).to(torch.bfloat16)
    rows = len(lens)
    perm = torch.randperm(num_pages - 1, generator=g)[: rows * pages_per_row] + 1
    bt = perm.view(rows, pages_per_row).to(torch.int32)
    return cache.to(DEV), bt.to(DEV)


@pytest.mark.parametrize("H", [16, 32, 128])
@pytest.mark.parametrize("lens", [[1], [17, 33, 1000, 5], [64] * 40, [1280, 31]])
def test_mla_decode(H, lens):
    cache, bt = _setup(lens)
    T = len(lens)
    q = (torch.randn(T, H, 576, device=DEV) * 0.3).to(torch.bfloat16)
    rows = torch.arange(T, dtype=torch.int32, device=DEV)
    kl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = ops.mla_attn(q, cache, bt, rows, kl, 0.0723)
    want = ref.mla_attn(q.cpu(), cache.cpu(), bt.cpu(), rows.cpu(), kl.cpu(), 0.0723)
    err = (out.float().cpu() - want.float()).abs().max().item()
    assert err < 2e-2, err


@pytest.mark.parametrize("H", [16, 64])
def test_mla_prefill_causal(H):
    # two sequences, chunked: seq 0 has 100 cached tokens + 150 new, seq 1 is a fresh 90-token prompt
    cache, bt = _setup([250, 90])
    q_lens, starts = [150, 90], [100, 0]
    tok_row, kv = [], []
    for s, (n, st) in enumerate(zip(q_lens, starts)):
        tok_row += [s] * n
        kv += [st + j + 1 for j in range(n)]
    T = len(tok_row)
    q = (torch.randn(T, H, 576, device=DEV) * 0.3).to(torch.bfloat16)
    rows = torch.tensor(tok_row, dtype=torch.int32, device=DEV)
    kl = torch.tensor(kv, dtype=torch.int32, device=DEV)
    out = ops.mla_attn(q, cache, bt, rows, kl, 0.0723)
    want = ref.mla_attn(q.cpu(), cache.cpu(), bt.cpu(), rows.cpu(), kl.cpu(), 0.0723)
    assert (out.float().cpu() - want.float()).abs().max().item() < 2e-2


@pytest.mark.parametrize("H", [40, 16, 8])
@pytest.mark.parametrize("lens", [[1], [17, 33, 1000, 5], [64] * 40])
def test_mla_minicpm3_shape(H, lens):
    """(kv_lora_rank 256 | rope 32) latent rows, head counts that are not a multiple of 16."""
    cache, bt = _setup(lens, dk=288)
    T = len(lens)
    q = (torch.randn(T, H, 288, device=DEV) * 0.3).to(torch.bfloat16)
    rows = torch.arange(T, dtype=torch.int32, device=DEV)
    kl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = ops.mla_attn(q, cache, bt, rows, kl, 0.0723, dv=256)
    want = ref.mla_attn(q.cpu(), cache.cpu(), bt.cpu(), rows.cpu(), kl.cpu(), 0.0723, 256)
    assert out.shape == (T, H, 256)
    assert (out.float().cpu() - want.float()).abs().max().item() < 2e-2


@pytest.mark.parametrize("mode,scoring", [(0, "softmax"), (1, "softmax"), (2, "sigmoid")])
def test_grouped_route(mode, scoring):
    torch.manual_seed(3)
    T, E = 300, 256
    logits = torch.randn(T, E, device=DEV) * 2
    bias = (torch.randn(E, device=DEV) * 0.05) if mode == 2 else None
    w, ids = ops.moe_route(logits, 8, True, scoring, bias=bias, n_group=8, topk_group=4, group_mode=mode)
    rw, rids = ref.moe_route(logits.cpu(), 8, True, scoring, bias.cpu() if bias is not None else None, 8, 4, mode)
    a = torch.sort(ids.cpu().long(), -1).values
    b = torch.sort(rids.long(), -1).values
    assert (a == b).float().mean().item() > 0.995
    assert torch.allclose(torch.sort(w.cpu(), -1).values, torch.sort(rw, -1).values, atol=1e-4)


def test_deepseek_engine_gpu():
    from ome_amd.runtime.engine import Engine, EngineArgs
    from ome_amd.runtime.request import SamplingParams

    eng = Engine(EngineArgs(model="tiny-deepseek", max_running_requests=8, context_length=512))
    rng = random.Random(0)
    prompts = [[rng.randrange(3, 1000) for _ in range(rng.randrange(3, 200))] for _ in range(6)]
    prompts.append(prompts[0])
    reqs = eng.generate(prompts, SamplingParams(max_new_tokens=16, temperature=0.0, ignore_eos=True))
    eng.flush()
    assert all(len(r.output_ids) == 16 for r in reqs)
    assert reqs[0].output_ids == reqs[-1].output_ids


def test_deepseek_gpu_vs_cpu_logits():
    from ome_amd.models import build_model
    from ome_amd.models.config import preset
    from tests.test_deepseek_cpu import _kv, _meta_prefill

    cfg = preset("tiny-deepseek")
    a = build_model(cfg, "cpu", torch.float32, load_format="dummy", seed=2)
    b = build_model(cfg, DEV, torch.bfloat16, load_format="dummy", seed=2)
    # same random weights on both devices (generators differ per device): copy CPU -> GPU
    for name, v in vars(a).items():
        if isinstance(v, list) and v and any(isinstance(t, torch.Tensor) for t in v):
            setattr(b, name, [t.to(DEV, torch.float32 if t.dtype == torch.float32 and name == "b_router"
                                   else torch.bfloat16) if isinstance(t, torch.Tensor) else t for t in v])
    for name in ("embed", "norm", "lm_head"):
        setattr(b, name, getattr(a, name).to(DEV, torch.bfloat16))
    ids = list(range(3, 40))
    la = a.compute_logits(a.forward(torch.tensor(ids, dtype=torch.int32), _meta_prefill(len(ids)), _kv(a)))
    meta = _meta_prefill(len(ids))
    for f in ("positions", "slots", "block_tables", "cu_q", "kv_lens", "items"):
        setattr(meta, f, getattr(meta, f).to(DEV))
    hk, dk, dv = b.kv_layout
    from ome_amd.models.common import PagedKVCache

    kvb = PagedKVCache(cfg.num_layers, 8, hk, dk, 16, torch.bfloat16, DEV, dv)
    lb = b.compute_logits(b.forward(torch.tensor(ids, dtype=torch.int32, device=DEV), meta, kvb)).float().cpu()
    cos = torch.nn.functional.cosine_similarity(la, lb, dim=-1)
    assert cos.min().item() > 0.99, cos.min()


@pytest.mark.parametrize("qlr,lat,rope,H,nope", [(1536, 512, 64, 16, 128), (768, 256, 32, 8, 64), (0, 512, 64, 4, 128)])
def test_mla_prep_matches_reference(qlr, lat, rope, H, nope):
    """Fused kv_a_layernorm + RoPE(k_pe) cache write + RoPE(q_pe) (``ome_mla_prep``) against the
    eager fp32 reference path, including a padding row (slot -1 -> scratch row 0)."""
    torch.manual_seed(qlr + lat)
    T, npos = 37, 4096
    a = torch.randn(T, qlr + lat + rope, dtype=torch.bfloat16)
    w = (1 + 0.1 * torch.randn(lat)).to(torch.bfloat16)
    q = torch.randn(T, H, nope + rope, dtype=torch.bfloat16)
    pos = torch.randint(0, npos, (T,), dtype=torch.int32)
    ang = torch.arange(npos)[:, None].float() * (1.0 / 10000 ** (torch.arange(0, rope, 2).float() / rope))[None]
    cs = torch.cat([ang.cos(), ang.sin()], -1).contiguous()
    slots = torch.randperm(200)[:T].to(torch.int32) + 1
    slots[5] = -1
    outs = []
    for dev in ("cpu", "cuda"):
        flat = torch.zeros(256, lat + rope, dtype=torch.bfloat16, device=dev)
        qf = torch.zeros(T, H, lat + rope, dtype=torch.bfloat16, device=dev)
        ops.mla_prep(a.to(dev), qlr, lat, rope, w.to(dev), 1e-6, pos.to(dev), cs.to(dev), slots.to(dev), flat,
                     q.to(dev), nope, qf)
        outs.append((flat.float().cpu(), qf.float().cpu()))
    (f0, q0), (f1, q1) = outs
    assert (f1 - f0).abs().max().item() <= 2e-2 * max(1.0, f0.abs().max().item())
    assert (q1[:, :, lat:] - q0[:, :, lat:]).abs().max().item() <= 2e-2 * max(1.0, q0.abs().max().item())
    assert f1[0].abs().sum() > 0   # the padding row landed in the scratch row


def _exact(q, cache, bt, rows, kl, scale):
    """Attention in 64 bits, token by token."""
    out = torch.zeros(q.shape[0], q.shape[1], 512, dtype=torch.float64)
    q, cache, bt = q.cpu().double(), cache.cpu().double().view(-1, 576), bt.cpu().long()
    for t, (r, n) in enumerate(zip(rows.tolist(), kl.tolist())):
        at = torch.arange(n)
        kv = cache[bt[r][at // 16] * 16 + at % 16]
        out[t] = (q[t] @ kv.T * scale).softmax(-1) @ kv[:, :512] if n else 0
    return out


@pytest.mark.parametrize("rows", [0, 32, 64, 128])
@pytest.mark.parametrize("H", [16, 20, 64, 128])
@pytest.mark.parametrize("seqs", [[(1, 1), (33, 33), (0, 40)], [(70, 9), (5, 3), (0, 1), (31, 34)], [(700, 30)]], ids=str)
def test_mla_row_tiles_of_prompts(monkeypatch, seqs, H, rows):
    """(cached tokens, new tokens) per sequence: tiles that end inside a token's heads, hold several sequences, or
    are cut into partitions; contexts around whole key tiles and pages."""
    torch.manual_seed(H)
    cache, bt = _setup([a + n for a, n in seqs])
    row = torch.tensor([s for s, (_, n) in enumerate(seqs) for _ in range(n)], dtype=torch.int32)
    kl = torch.tensor([a + j + 1 for a, n in seqs for j in range(n)], dtype=torch.int32)
    q = torch.randn(len(row), H, 576, device=DEV).to(torch.bfloat16)
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (rows, False, ops.MLAWorkspace.parts(T, H, DK, rows)))
    out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 0.06)
    want = _exact(q, cache, bt, row, kl, 0.06)
    # probabilities and the output are rounded to bf16 once each: 2^-9 of the largest value they sum, and of the result
    assert (out.cpu().double() - want).abs().max() < 2.0 ** -8 * cache.float().abs().max().item()


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("scale", [0.06, -0.06, 0.0])
def test_mla_row_tiles_of_long_contexts(monkeypatch, rows, decode, scale):
    """Pieces of 31 to 66 key tiles: the pages are looked up 32 tiles at a time and moves run three ahead of the products.
    Scales that the row tiles leave to the 16-head kernel."""
    torch.manual_seed(rows)
    new = [1] * 5 if decode else [2, 5, 3]
    ctx = [980, 1024, 1056, 1057, 2100][:len(new)]
    cache, bt = _setup([a + n for a, n in zip(ctx, new)])
    row = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32)
    kl = torch.tensor([a + j + 1 for a, n in zip(ctx, new) for j in range(n)], dtype=torch.int32)
    q = torch.randn(len(row), 16, 576, device=DEV).to(torch.bfloat16)
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (rows, decode, 1))
    out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), scale)
    want = _exact(q, cache, bt, row, kl, scale)
    assert (out.cpu().double() - want).abs().max() < 2.0 ** -8 * cache.float().abs().max().item()


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("H", [16, 32, 64, 128])
@pytest.mark.parametrize("lens", [[1, 0, 32, 33], [5000, 16, 700], [200, 31, 64, 65, 1] * 13, [40] * 260, list(range(1, 257))],
                         ids=lambda v: f"{len(v)}x{max(v)}")
def test_mla_row_tiles_of_decode_steps(monkeypatch, lens, H, rows):
    """Contexts cut by length into at most 256 pieces: empty and single-key ones, one long among short, as many tokens
    as pieces, more."""
    torch.manual_seed(len(lens))
    cache, bt = _setup(lens)
    q = torch.randn(len(lens), H, 576, device=DEV).to(torch.bfloat16)
    row, kl = torch.arange(len(lens), dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (rows, True, ops.MLAWorkspace.parts(T, H, DK, rows, True)))
    out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 0.06)
    want = _exact(q, cache, bt, row, kl, 0.06)
    assert (out.cpu().double() - want).abs().max() < 2.0 ** -8 * cache.float().abs().max().item()


@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("H", [20, 128])
@pytest.mark.parametrize("first,pad", [(0, 64), (8, 8), (1, 0), (0, 4)], ids=str)
def test_mla_row_tiles_take_queries_of_any_stride(monkeypatch, decode, H, first, pad):
    """Rows that start on 16 bytes come by way of LDS, others straight into registers: the same bits; outputs of a wider row too."""
    torch.manual_seed(H + first)
    new = [1] * 9 if decode else [11, 3, 20]
    cache, bt = _setup([40 + n for n in new])
    row = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32, device=DEV)
    kl = torch.tensor([40 + j + 1 for n in new for j in range(n)], dtype=torch.int32, device=DEV)
    T = len(row)
    wide = torch.randn(T * (H * 576 + pad) + 16, device=DEV).to(torch.bfloat16)
    q = wide[first:first + T * (H * 576 + pad)].view(T, H * 576 + pad)[:, :H * 576].unflatten(1, (H, 576))
    out = torch.empty(T, H * 512 + 24, dtype=torch.bfloat16, device=DEV)[:, :H * 512].unflatten(1, (H, 512))
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (128, decode, 2 if decode else 1))
    want = ops.mla_attn(q.contiguous(), cache, bt, row, kl, 0.06)
    assert torch.equal(ops.mla_attn(q, cache, bt, row, kl, 0.06, out=out), want)


def test_mla_tile_rule_fits_workspace_and_chip():
    """Tiles of prompts fill at most one launch wave when partitioned; partials fit the workspace."""
    W = ops.MLAWorkspace
    for H in (4, 16, 20, 64, 128):
        for T in (1, 3, 4, 7, 30, 63, 64, 200, 700, 5000):
            for seqs in (1, 2, 7, 64, 600):
                for pages in (1, 2, 16, 17, 64, 65, 1024):
                    rows, decode, parts = W.tiles(T, H, 576, seqs, pages)
                    assert rows in (0, 32, 64, 128) and parts >= 1 and (rows or not decode)
                    if rows and not decode and parts > 1:
                        wgs = -(-T * H // rows)
                        assert wgs * parts <= W.TARGET_WGS_ALL and wgs * rows * parts <= W.ROWS
                    assert W.tiles(T, H, 288, seqs, pages)[0] == 0


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("H,parts", [(16, 1), (16, 3), (64, 1)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_mla_row_tiles_keep_a_broken_sequence_apart(monkeypatch, rows, H, parts, bad):
    """Latents of one sequence that are not finite: the others, whose rows share tiles with it, stay what they were, bit
    for bit."""
    torch.manual_seed(rows + H)
    new = [5, 1, 37, 3, 20]
    cache, bt = _setup([40 + n for n in new])
    row = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32, device=DEV)
    kl = torch.tensor([40 + j + 1 for n in new for j in range(n)], dtype=torch.int32, device=DEV)
    q = torch.randn(len(row), H, 576, device=DEV).to(torch.bfloat16)
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (rows, False, parts))
    want = ops.mla_attn(q, cache, bt, row, kl, 0.06)
    for s in (1, 3):
        cache[bt[s].long()[:2], :, ::7] = bad
    got = ops.mla_attn(q, cache, bt, row, kl, 0.06)
    whole = (row != 1) & (row != 3)
    assert torch.equal(got[whole], want[whole]) and not got[~whole].isfinite().all()


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("H,parts", [(16, 1), (20, 2), (64, 1)])
def test_mla_row_tiles_take_tokens_in_any_order(monkeypatch, rows, H, parts):
    torch.manual_seed(rows + H)
    new = [9, 2, 0, 30, 1, 6]
    cache, bt = _setup([30 + n for n in new])
    row = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32)
    kl = torch.tensor([30 + j + 1 for n in new for j in range(n)], dtype=torch.int32)
    at = torch.randperm(len(row))
    row, kl = row[at], kl[at]
    q = torch.randn(len(row), H, 576, device=DEV).to(torch.bfloat16)
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (rows, False, parts))
    out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 0.06)
    assert (out.cpu().double() - _exact(q, cache, bt, row, kl, 0.06)).abs().max() < 2.0 ** -8 * cache.float().abs().max().item()


@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("rows,H", [(32, 16), (64, 64), (128, 128)])
def test_mla_row_tiles_are_as_exact_as_the_16_head_kernel(monkeypatch, rows, H, decode):
    """Error against 64 bits, of scores as wide as DeepSeek's (1.7 in natural units).  Both kernels round weights and
    outputs to bf16; the 16-head kernel's largest weight of a row is exactly 1, a row tile's is used in two parts.  2% for
    the other order of rounding."""
    torch.manual_seed(H)
    new = [1] * 24 if decode else [110, 60]
    ctx = [800 + 70 * i for i in range(24)] if decode else [1100, 260]
    cache, bt = _setup(ctx)
    row = torch.tensor([s for s, n in enumerate(new) for _ in range(n)], dtype=torch.int32)
    kl = torch.tensor([c - n + j + 1 for c, n in zip(ctx, new) for j in range(n)], dtype=torch.int32)
    q = torch.randn(len(row), H, 576, device=DEV).to(torch.bfloat16)
    want = _exact(q, cache, bt, row, kl, 2 * 192 ** -0.5)
    err = []
    for tile in (0, rows):
        monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda T, H, DK, *a: (tile, decode and tile > 0, ops.MLAWorkspace.parts(
            T, H, DK, tile, decode and tile > 0)))
        out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 2 * 192 ** -0.5).cpu().double()
        err.append(((out - want).norm() / want.norm()).item())
    assert err[1] < 1.02 * err[0], err


@pytest.mark.parametrize("T,H", [(1, 16), (3, 32), (7, 40), (15, 16)])
def test_mla_partitions_by_length(T, H):
    """Few decode rows: partitions of up to four key tiles and more, empty ones, contexts at the edges of both.  bf16 weights and outputs:
    two roundings of 2^-9."""
    torch.manual_seed(T)
    every = [1, 31, 32, 33, 127, 511, 512, 513, 1537, 2047, 2048, 2049, 3000, 5000, 8193]
    for at in range(0, len(every), T):
        ctx = (every[at:] + every)[:T]
        cache, bt = _setup(ctx)
        row, kl = torch.arange(T, dtype=torch.int32), torch.tensor(ctx, dtype=torch.int32)
        q = torch.randn(T, H, 576, device=DEV).to(torch.bfloat16)
        want = _exact(q, cache, bt, row, kl, 192 ** -0.5)
        out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 192 ** -0.5).cpu().double()
        assert ((out - want).flatten(1).norm(dim=1) <= 2.0 ** -8 * want.flatten(1).norm(dim=1)).all(), ctx


@pytest.mark.parametrize("T,H", [(20, 16), (11, 24), (40, 8)])
@pytest.mark.parametrize("longest", [48, 230, 1100, 4500])
def test_mla_waves_with_pages_of_their_own(T, H, longest):
    """Contexts at the edges of pages, of a page for each wave and of 64 of a wave's pages, in one partition and in several, over a cache whose rows
    past the contexts are NaN.  Tolerance as above."""
    torch.manual_seed(T)
    every = [n for n in (longest, 0, 1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 128, 129, 240, 513, 1024, 1090, 4096, 4097) if n <= longest]
    ctx = (every * T)[:T]
    cache, bt = _setup(ctx)
    for s, n in enumerate(ctx):
        if n % 16:
            cache[bt[s, n // 16].item(), n % 16:] = float("nan")
    row, kl = torch.arange(T, dtype=torch.int32), torch.tensor(ctx, dtype=torch.int32)
    q = torch.randn(T, H, 576, device=DEV).to(torch.bfloat16)
    assert ops.MLAWorkspace.parts(T, H, 576, pages=bt.shape[1]) == {48: 1, 230: 4}.get(longest, 256 // (T * -(-H // 16)))
    for parts in (None, 1, 3):
        with pytest.MonkeyPatch.context() as mp:
            p = parts or ops.MLAWorkspace.parts(T, H, 576, pages=bt.shape[1])
            mp.setattr(ops.MLAWorkspace, "tiles", lambda *a: (0, False, p))
            out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 192 ** -0.5).cpu().double()
        want = _exact(q, torch.nan_to_num(cache), bt, row, kl, 192 ** -0.5)
        live = kl > 0
        assert bool((out[~live] == 0).all())
        assert ((out - want).flatten(1).norm(dim=1)[live] <= 2.0 ** -8 * want.flatten(1).norm(dim=1)[live]).all()


@pytest.mark.parametrize("H", [4, 9, 16])
@pytest.mark.parametrize("lens,parts", [([1, 0, 32, 33, 5000], 52), (list(range(1, 257)), 1), ([700, 16, 64, 65, 1] * 13, 8), ([4097, 0] * 12, 22), ([300] * 200, 3)], ids=str)
def test_mla_pieces_by_length_of_few_heads(monkeypatch, lens, parts, H):
    """Decode steps of up to 16 heads over wide tables, with pieces of no, one and many pages and none at all, NaN in the workspace and past the contexts, at half the bound
    above: weights are exact to 2^-17."""
    torch.manual_seed(H)
    cache, bt = _setup(lens)
    for s, n in enumerate(lens):
        if n % 16:
            cache[bt[s, n // 16].item(), n % 16:] = float("nan")
    bt = torch.nn.functional.pad(bt, (0, max(0, 3000 // len(lens) + 1 - bt.shape[1])))
    row, kl = torch.arange(len(lens), dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    q = torch.randn(len(lens), H, 576, device=DEV).to(torch.bfloat16)
    ws = ops.MLAWorkspace(DEV)
    ws.ws_o.fill_(float("nan"))
    ws.ws_ml.fill_(float("nan"))
    monkeypatch.setattr(ops.MLAWorkspace, "tiles", lambda *a: (32, True, parts))
    out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 192 ** -0.5, ws).cpu().double()
    want = _exact(q, torch.nan_to_num(cache), bt, row, kl, 192 ** -0.5)
    assert bool((out[kl == 0] == 0).all())
    assert ((out - want).flatten(1).norm(dim=1) <= 2.0 ** -9 * want.flatten(1).norm(dim=1)).all()


@pytest.mark.parametrize("T,H", [(1, 16), (3, 32), (12, 16)])
def test_mla_reads_no_partition_that_is_not_written(T, H):
    """A workspace that holds NaN, contexts of fewer partitions than the table's width allows, and the tokens' own lengths.  Tolerance as above."""
    torch.manual_seed(T)
    for every in ([0, 1, 300, 511], [513, 2048, 2049, 2500], [3000, 4097, 8000, 0]):
        ctx = (every * T)[:T]
        cache, bt = _setup(ctx + [8192])
        row, kl = torch.arange(T, dtype=torch.int32), torch.tensor(ctx, dtype=torch.int32)
        q = torch.randn(T, H, 576, device=DEV).to(torch.bfloat16)
        ws = ops.MLAWorkspace(DEV)
        ws.ws_o.fill_(float("nan"))
        ws.ws_ml.fill_(float("nan"))
        assert ops.MLAWorkspace.tiles(T, H, 576, *bt.shape)[2] > 16
        out = ops.mla_attn(q, cache, bt, row.to(DEV), kl.to(DEV), 192 ** -0.5, ws).cpu().double()
        for t, n in enumerate(ctx):
            if n == 0:
                assert bool((out[t] == 0).all())
                continue
            want = _exact(q[t:t + 1], cache, bt[t:t + 1], row[:1], kl[t:t + 1], 192 ** -0.5)
            assert ((out[t:t + 1] - want).flatten(1).norm(dim=1) <= 2.0 ** -8 * want.flatten(1).norm(dim=1)).all(), (ctx, t)


@pytest.mark.parametrize("pages,most", [(20, 16), (128, 16), (129, 64)])
@pytest.mark.parametrize("window", [0, 4096])
def test_latent_partitions_with_sinks_go_by_the_tables_width(monkeypatch, pages, most, window):
    """Sinks and windows, which take the 16-head kernel: no more partitions than a table of that width is worth.  Tolerance as above."""
    torch.manual_seed(pages)
    n = 16 * pages - 5
    cache, bt = _setup([16 * (pages - 1)])
    assert bt.shape[1] == pages
    q, sinks = torch.randn(1, 16, 576, device=DEV).to(torch.bfloat16), torch.randn(16, device=DEV)
    row, kl = torch.zeros(1, dtype=torch.int32, device=DEV), torch.tensor([n], dtype=torch.int32, device=DEV)
    parts, call = [], ops.call
    monkeypatch.setattr(ops, "call", lambda fn, *a: (parts.append(a[13]), call(fn, *a)))
    out = ops.latent_attn(q, cache, bt, row, kl, 192 ** -0.5, 512, sinks=sinks, window=window).cpu().double()
    assert parts == [min(most, window // 128 if window else most)]
    at = torch.arange(max(0, n - window) if window else 0, n)
    kv = cache.cpu().double().view(-1, 576)[bt[0].cpu().long()[at // 16] * 16 + at % 16]
    s = torch.cat([q[0].cpu().double() @ kv.T * 192 ** -0.5, sinks.cpu().double()[:, None]], 1).softmax(-1)[:, :-1]
    want = s @ kv[:, :512]
    assert (out[0] - want).norm() <= 2.0 ** -8 * want.norm()
