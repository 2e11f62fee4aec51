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


@pytest.mark.parametrize("K", [2, 3, 4, 5, 6, 7])
def test_short_conv_in_place(K):
    """The output may be the input: the same sums in the same order (7 taps: another exponential, one bf16 rounding)."""
    torch.manual_seed(1)
    sq, C = seqs([40, 1, 19], 4), 264
    x, w, st = torch.randn(60, C, device=DEV).to(BF), torch.randn(C, K, device=DEV).to(BF), torch.randn(4, C, K - 1, device=DEV).to(BF)
    s2 = st.clone()
    want = ops.ssm_conv1d(x, w, None, st, *sq)
    got = ops.ssm_conv1d(x, w, None, s2, *sq, out=x)
    assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=1e-5) and torch.equal(st, s2)
    assert K > 6 or torch.equal(got, want)


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


def exact_gdn(q, k, v, a, b, A_log, dtb, state, cu, slot, reset, Hv, Hk):
    q, k, v, a, b, A_log, dtb = (t.cpu().double() for t in (q, k, v, a, b, A_log, dtb))
    st, dv, dk = state.cpu().double(), state.shape[2], state.shape[3]
    unit = lambda t: t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt()  # noqa: E731
    out = torch.zeros(q.shape[0], Hv, dv, dtype=torch.float64)
    for s, sl in enumerate(slot.tolist()):
        r0, r1 = cu[s:s + 2].tolist()
        S = st[sl] * (0.0 if reset[s] else 1.0)
        for r in range(r0, r1):
            kr = unit(k[r].view(Hk, dk)).repeat_interleave(Hv // Hk, 0)
            qr = unit(q[r].view(Hk, dk)).repeat_interleave(Hv // Hk, 0) * dk ** -0.5
            S = S * torch.exp(-A_log.exp() * torch.nn.functional.softplus(a[r] + dtb))[:, None, None]
            u = (v[r].view(Hv, dv) - (S @ kr[:, :, None])[..., 0]) * b[r].sigmoid()[:, None]
            S = S + u[:, :, None] * kr[:, None]
            out[r] = (S @ qr[:, :, None])[..., 0]
        if r1 > r0:
            st[sl] = S
    return out.flatten(1), st


def exact_ssm(x, dt, B, C, A, D, dtb, dt_min, state, cu, slot, reset, H, P, N, G):
    x, dt, B, C, A, D, dtb = (t.cpu().double() for t in (x, dt, B, C, A, D, dtb))
    st = state.cpu().double()
    out = torch.zeros(x.shape[0], H, P, dtype=torch.float64)
    for s, sl in enumerate(slot.tolist()):
        r0, r1 = cu[s:s + 2].tolist()
        S = st[sl] * (0.0 if reset[s] else 1.0)
        for r in range(r0, r1):
            d = torch.nn.functional.softplus(dt[r] + dtb).clamp(min=dt_min)
            b, c = (t[r].view(G, N).repeat_interleave(H // G, 0) for t in (B, C))
            S = S * (d * A).exp()[:, None, None] + (d[:, None] * x[r].view(H, P))[:, :, None] * b[:, None]
            out[r] = (S @ c[:, :, None])[..., 0] + D[:, None] * x[r].view(H, P)
        if r1 > r0:
            st[sl] = S
    return out.flatten(1), st


def near(out, state, want, want_state):
    """Outputs: one rounding to bf16 (2^-9 of each value at most, so of the whole).  States: fp32 sums; a state row is a
    sum of at most 2^8 products whose weights (decays, norms) carry a few fp32 roundings each: 2^-24 * 2^5."""
    rel = lambda x, y: ((x.cpu().double() - y).norm() / y.norm()).item()  # noqa: E731
    return rel(out, want) < 2.0 ** -9 and rel(state, want_state) < 2.0 ** -19


@pytest.mark.parametrize("lens", LENS, ids=str)
@pytest.mark.parametrize("dk,dv,Hk,Hv,off", [(128, 128, 2, 4, 8), (64, 16, 1, 5, 0), (128, 80, 3, 3, 8), (64, 128, 2, 2, 1)])
def test_delta_rule_prompts(lens, dk, dv, Hk, Hv, off):
    torch.manual_seed(dk + dv)
    T, slots, kd, vd = sum(lens), 71, Hk * dk, Hv * dv
    c = torch.randn(T, 2 * kd + vd + off, device=DEV).to(BF)[:, off:]   # off 1: the row-by-row kernel
    ab = torch.randn(T, 2 * Hv, device=DEV).to(BF)
    A_log, dtb = torch.linspace(-4, 2.5, Hv, device=DEV), torch.randn(Hv, device=DEV)
    st = torch.randn(slots, Hv, dv, dk, device=DEV) * 0.2
    sq = seqs(lens, slots)
    args = (c[:, :kd], c[:, kd:2 * kd], c[:, 2 * kd:], ab[:, :Hv], ab[:, Hv:], A_log, dtb)
    want = exact_gdn(*args, st, *sq, Hv, Hk)
    assert near(ops.gdn_scan(*args, st, *sq, Hv, Hk), st, *want)


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("dv,shift,gap", [(128, 1, 0), (16, 8, 4), (80, 0, 2), (48, 0, 1), (64, 8, 0)])
def test_chunked_scans_of_values_and_outputs_of_any_alignment(dv, shift, gap, delta):
    """Keys and queries that the chunks take, values ``shift`` columns and outputs ``gap`` columns further in their rows: pieces of
    16 and 8 bytes where both are aligned for them, single values elsewhere; columns that fill no block of 64."""
    torch.manual_seed(dv + shift)
    lens, H, dk = [40, 0, 7, 65], 2, 128
    T, kd, sq = sum(lens), H * dk, seqs(lens, 71)
    c, ab = torch.randn(T, 2 * kd + H * dv + 16, device=DEV).to(BF), torch.randn(T, 2 * H, device=DEV).to(BF)
    q, k, v = c[:, :kd], c[:, kd:2 * kd], c[:, 2 * kd + shift:2 * kd + shift + H * dv]
    out = torch.full((T, H * dv + 2 * gap), 7.0, device=DEV).to(BF)
    o, st, bias = out[:, gap:gap + H * dv], torch.randn(71, H, dv, dk, device=DEV) * 0.2, torch.randn(H, device=DEV)
    if delta:
        args = (q, k, v, ab[:, :H], ab[:, H:], torch.linspace(-3, 2, H, device=DEV), bias)
        want = exact_gdn(*args, st, *sq, H, H)
        ops.gdn_scan(*args, st, *sq, H, H, out=o)
    else:
        args = (v, ab[:, :H], k, q, -torch.logspace(-1, 1, H, device=DEV), torch.randn(H, device=DEV), bias, 0.001)
        want = exact_ssm(*args, st, *sq, H, dv, dk, H)
        ops.ssm_scan(*args, st, *sq, H, dv, dk, H, out=o)
    assert near(o, st, *want)
    assert bool((out[:, :gap] == 7).all()) and bool((out[:, gap + H * dv:] == 7).all())


@pytest.mark.parametrize("lens", [[1], [1] * 5, [1, 0, 2, 1], [1] * 70], ids=str)
@pytest.mark.parametrize("dk,dv,Hk,Hv,off", [(128, 128, 2, 4, 8), (64, 16, 1, 5, 0), (256, 40, 3, 3, 8), (128, 33, 1, 2, 8),
                                             (64, 128, 2, 2, 1)])
def test_delta_rule_steps(lens, dk, dv, Hk, Hv, off):   # off 1: the scan behind its prep pass
    test_delta_rule_prompts(lens, dk, dv, Hk, Hv, off)


@pytest.mark.parametrize("lens", LENS, ids=str)
@pytest.mark.parametrize("H,P,N,G,off", [(16, 64, 128, 2, 8), (3, 16, 64, 1, 0), (5, 80, 128, 5, 8), (4, 64, 128, 2, 1),
                                         (20, 16, 64, 2, 8)])
def test_selective_scan_prompts(lens, H, P, N, G, off):
    torch.manual_seed(H + N)
    T, slots = sum(lens), 71
    c = torch.randn(T, H * P + 2 * G * N + off, device=DEV).to(BF)[:, off:]
    dt = torch.randn(T, H + 3, device=DEV).to(BF)[:, 3:]
    A, D, dtb = -torch.logspace(-1, 1.2, H, device=DEV), torch.randn(H, device=DEV), torch.linspace(-6, 1, H, device=DEV)
    st = torch.randn(slots, H, P, N, device=DEV) * 0.2
    sq = seqs(lens, slots)
    args = (c[:, :H * P], dt, c[:, H * P:H * P + G * N], c[:, H * P + G * N:], A, D, dtb, 0.001)
    want = exact_ssm(*args, st, *sq, H, P, N, G)
    assert near(ops.ssm_scan(*args, st, *sq, H, P, N, G), st, *want)


@pytest.mark.parametrize("rows", [5, 31, 32, 64])
@pytest.mark.parametrize("N", [64, 128])
def test_selective_scan_entry_by_entry(rows, N):
    """Values that are 1 in a column of their own: the output is exp(cum_i - cum_j) dt_j q_i.k_j, each entry by itself, zero above the diagonal."""
    torch.manual_seed(rows + N)
    H, P = 2, 64
    B, C = (torch.randn(rows, N, device=DEV).to(BF) for _ in range(2))
    dt = torch.randn(rows, H, device=DEV).to(BF)
    x = torch.eye(rows, P, device=DEV).to(BF).repeat(1, H)
    A, D, dtb = torch.tensor([-0.02, -1.5], device=DEV), torch.zeros(H, device=DEV), torch.zeros(H, device=DEV)
    state = torch.zeros(1, H, P, N, device=DEV)
    out = ops.ssm_scan(x, dt, B, C, A, D, dtb, 0.0, state, i32([0, rows]), i32([0]), i32([1]), H, P, N, 1).view(rows, H, P).transpose(0, 1)
    step = torch.nn.functional.softplus(dt.double().T)   # [H, rows]
    cum = (step * A.double()[:, None]).cumsum(1)
    want = torch.exp(cum[:, :, None] - cum[:, None, :]) * step[:, None, :] * (C.double() @ B.double().T)
    want = torch.nn.functional.pad(want.tril(), (0, P - rows))
    size = torch.nn.functional.pad(((C.double().abs() @ B.double().abs().T) * step[:, None, :]).tril(), (0, P - rows))
    # rounded to bf16 once, of 8 bits: half a step is 2^-8 of a value at the most; fp32 sums of up to 128 products before it
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * size).all())


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("what", ["q", "k", "v", "a", "b"])
def test_delta_rule_stays_causal(what, bad):
    """A value that is not finite reaches its own row and the rows after it, of its heads: nothing earlier in its chunk."""
    torch.manual_seed(5)
    lens, Hk, Hv, dk, dv, at = [40, 90, 33], 2, 4, 64, 32, 40 + 43   # row 11 of the second sequence's second chunk
    T, kd, sq = sum(lens), Hk * dk, (i32([0, 40, 130, 163]), i32([0, 1, 2]), i32([0, 1, 0]))
    t = {n: torch.randn(T, w, device=DEV).to(BF) for n, w in (("c", 2 * kd + Hv * dv), ("ab", 2 * Hv))}
    t.update(q=t["c"][:, :kd], k=t["c"][:, kd:2 * kd], v=t["c"][:, 2 * kd:], a=t["ab"][:, :Hv], b=t["ab"][:, Hv:])
    A_log, dtb, st = torch.linspace(-3, 1, Hv, device=DEV), torch.zeros(Hv, device=DEV), torch.randn(3, Hv, dv, dk, device=DEV)
    run = lambda s: ops.gdn_scan(t["q"], t["k"], t["v"], t["a"], t["b"], A_log, dtb, s, *sq, Hv, Hk).float().view(T, Hv, dv)  # noqa: E731
    s0, s1 = st.clone(), st.clone()
    clean = run(s0)
    t[what][at, 1] = bad   # the first key head (value heads 0, 1), head 0's column 1, head 1's gates
    heads = {"q": [0, 1], "k": [0, 1], "v": [0], "a": [1], "b": [1]}[what]
    got = run(s1)
    hit = torch.zeros_like(clean, dtype=torch.bool)
    hit[at:130, heads] = True
    # another path's sums for the rows of its chunk: one bf16 step of the largest value
    assert (got - clean)[~hit].abs().max() <= 2.0 ** -8 * clean.abs().max()
    assert torch.equal(s0[[0, 2]], s1[[0, 2]])
    want_out = torch.empty(T, Hv * dv, dtype=torch.float32)
    want_st = st.cpu()
    ref.gdn_scan(*cpu(t["q"], t["k"], t["v"], t["a"], t["b"], A_log, dtb), want_st, *cpu(*sq), Hv, Hk, want_out)
    assert torch.equal(s1.cpu().isfinite(), want_st.isfinite())


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("what", ["x", "dt", "B", "C"])
def test_selective_scan_stays_causal(what, bad):
    torch.manual_seed(6)
    lens, H, P, N, G, at = [40, 90, 33], 4, 32, 64, 2, 40 + 43
    T, sq = sum(lens), (i32([0, 40, 130, 163]), i32([0, 1, 2]), i32([0, 1, 0]))
    t = {n: torch.randn(T, w, device=DEV).to(BF) for n, w in (("x", H * P), ("dt", H), ("bc", 2 * G * N))}
    t.update(B=t["bc"][:, :G * N], C=t["bc"][:, G * N:])
    A, D, dtb = -torch.logspace(-1, 1, H, device=DEV), torch.randn(H, device=DEV), torch.linspace(-4, 0, H, device=DEV)
    st = torch.randn(3, H, P, N, device=DEV)
    run = lambda s: ops.ssm_scan(t["x"], t["dt"], t["B"], t["C"], A, D, dtb, 0.001, s, *sq, H, P, N, G).float().view(T, H, P)  # noqa: E731
    s0, s1 = st.clone(), st.clone()
    clean = run(s0)
    t[what][at, 1] = bad
    got = run(s1)
    hit = torch.zeros_like(clean, dtype=torch.bool)
    hit[at:130, {"x": [0], "dt": [1], "B": [0, 1], "C": [0, 1]}[what]] = True
    assert (got - clean)[~hit].abs().max() <= 2.0 ** -8 * clean.abs().max()
    assert torch.equal(s0[[0, 2]], s1[[0, 2]])


@pytest.mark.parametrize("delta", [True, False])
def test_scans_in_place_of_their_values(delta):
    """... as elsewhere, with a value that is not finite in the second of three sequences."""
    torch.manual_seed(7)
    H, dk, dv, lens, at = 4, 64, 32, [40, 90, 33], 40 + 43
    T, sq = sum(lens), (i32([0, 40, 130, 163]), i32([0, 1, 2]), i32([0, 1, 0]))
    c, ab = torch.randn(T, 2 * H * dk + H * dv, device=DEV).to(BF), torch.randn(T, 2 * H, device=DEV).to(BF)
    c[at, 2 * H * dk + 1] = float("nan")
    A, D, dtb, st = torch.linspace(-2, -0.1, H, device=DEV), torch.ones(H, device=DEV), torch.zeros(H, device=DEV), torch.randn(3, H, dv, dk, device=DEV)

    def run(s, out):
        q, k, v = c[:, :H * dk], c[:, H * dk:2 * H * dk], c[:, 2 * H * dk:]
        if delta:
            return ops.gdn_scan(q, k, v, ab[:, :H], ab[:, H:], A, dtb, s, *sq, H, H, out=out)
        return ops.ssm_scan(v, ab[:, :H], k, q, A, D, dtb, 0.001, s, *sq, H, dv, dk, H, out=out)

    s0, s1 = st.clone(), st.clone()
    want = run(s0, None).float()
    got = run(s1, c[:, 2 * H * dk:]).float()
    # another path's sums: one bf16 step of the largest value; states in fp32, of the same order
    assert torch.equal(got.isfinite(), want.isfinite()) and (got - want).nan_to_num(0.0).abs().max() <= 2.0 ** -8 * want.nan_to_num(0.0).abs().max()
    assert torch.equal(s0.isfinite(), s1.isfinite()) and (s0 - s1).nan_to_num(0.0).abs().max() <= 1e-5 * st.abs().max()


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("lens", [[1] * 3 + [40] + [1] * 60, [3, 4, 0, 2, 33, 1, 5, 32], [2] * 33], ids=str)
def test_decode_rows_beside_prompts_take_no_chunks(lens, delta, monkeypatch):
    """Sequences of up to three rows are walked row by row: their chunks of the workspace stay untouched."""
    kept = []

    def poisoned(*a):
        kept.append(make(*a).fill_(-7.0))
        return kept[0]

    make = ops._chunk_rule_ws
    monkeypatch.setattr(ops, "_chunk_rule_ws", poisoned)
    (test_delta_rule_prompts(lens, 128, 80, 3, 3, 8) if delta else test_selective_scan_prompts(lens, 16, 64, 128, 2, 8))
    ws, r0 = kept[0].view(sum(lens) // 32 + len(lens), -1), 0
    for s, n in enumerate(lens):
        if n:
            assert bool((ws[r0 // 32 + s] == -7.0).all()) == (n <= 3), (s, n)
        r0 += n


def test_few_rows_take_the_row_by_row_kernels():
    def ws(T, S, delta):
        c = torch.empty(T, 512, dtype=BF, device=DEV)
        st = torch.empty(S, 2, 64, 128, device=DEV)
        return ops._chunk_rule_ws(T, S, 2, 2, 128, 64, delta, st, (c[:, :256], c[:, 256:], c, torch.empty_like(c)))

    for delta, few in ((True, 32), (False, 4)):
        assert ws(few, 1, delta) is None and ws(few, 2, delta) is None and ws(40, 40, delta) is None
        assert ws(few + 1, 1, delta) is not None and ws(41, 40, delta) is not None


# segments of one chunk and more, whole and not, beside sequences of one segment, a few rows and none
@pytest.mark.parametrize("seg", [1, 2, 3])
@pytest.mark.parametrize("lens", [[97], [3, 0, 64, 65], [32, 160, 1, 96], [33, 2, 129]], ids=str)
@pytest.mark.parametrize("delta", [True, False])
def test_scans_in_segments(lens, seg, delta, monkeypatch):
    monkeypatch.setattr(ops, "_chunk_rule_seg", lambda *a: seg)
    if delta:
        for dims in ((128, 128, 2, 4, 8), (64, 16, 1, 5, 0), (128, 80, 3, 3, 8), (64, 128, 2, 2, 8)):
            test_delta_rule_prompts(lens, *dims)
    else:
        for dims in ((16, 64, 128, 2, 8), (3, 16, 64, 1, 0), (5, 80, 128, 5, 8), (2, 144, 64, 2, 8)):
            test_selective_scan_prompts(lens, *dims)


@pytest.mark.parametrize("seg", [0, 1, 2])
@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("delta", [True, False])
def test_many_workgroups_as_few(delta, dk, seg, monkeypatch):
    """Chunks moved by waves of their own (up to 256 workgroups) or by those that compute (more): the same bits."""
    monkeypatch.setattr(ops, "_chunk_rule_seg", lambda *a: seg)
    torch.manual_seed(dk + seg)
    lens, H, dv = [31, 3, 97, 0, 64, 1, 33], 96, 64
    T, sq = sum(lens), seqs(lens, 8)
    q, k, v = (torch.randn(T, H * d, device=DEV).to(BF) for d in (dk, dk, dv))
    ab, st = torch.randn(2, T, H, device=DEV).to(BF), torch.randn(8, H, dv, dk, device=DEV)
    A, zero = torch.linspace(-3, 0, H, device=DEV), torch.zeros(H, device=DEV)

    def scan(n):
        s = st[:, :n].clone()
        if delta:
            o = ops.gdn_scan(q[:, :n * dk], k[:, :n * dk], v.as_strided((T, n * dv), (H * dk, 1)), ab[0, :, :n], ab[1, :, :n], A[:n], zero[:n], s, *sq, n, n)
        else:
            o = ops.ssm_scan(v[:, :n * dv], ab[0, :, :n], k[:, :n * dk], q[:, :n * dk], -A[:n].exp(), zero[:n], zero[:n], 0.001, s, *sq, n, dv, dk, n)
        return o, s

    if delta:   # (values share the row stride of q and k)
        v = torch.randn(T, H * dk, device=DEV).to(BF)
    (o, s), (few, s2) = scan(H), scan(2)
    assert torch.equal(o[:, :2 * dv], few) and torch.equal(s[:, :2], s2)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("what", ["q", "k", "v", "a", "b"])
def test_delta_rule_in_segments_stays_causal(what, bad, monkeypatch):
    monkeypatch.setattr(ops, "_chunk_rule_seg", lambda *a: 1)
    test_delta_rule_stays_causal(what, bad)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("what", ["B", "C", "x", "dt"])
def test_selective_scan_in_segments_stays_causal(what, bad, monkeypatch):
    monkeypatch.setattr(ops, "_chunk_rule_seg", lambda *a: 1)
    test_selective_scan_stays_causal(what, bad)


@pytest.mark.parametrize("what", ["k", "v", "a", "b", "state"])
def test_not_finite_in_segments_as_in_one_piece(what, monkeypatch):
    """What follows a value that is not finite, over several segments: the same infinities and NaN."""
    torch.manual_seed(3)
    T, dk, dv, H = 200, 64, 32, 2
    c, ab = torch.randn(T, H * (2 * dk + dv), device=DEV).to(BF), torch.randn(T, 2 * H, device=DEV).to(BF)
    q, k, v, a, b = c[:, :H * dk], c[:, H * dk:2 * H * dk], c[:, 2 * H * dk:], ab[:, :H], ab[:, H:]
    st = torch.randn(1, H, dv, dk, device=DEV)
    (st[0, 0, 5] if what == "state" else {"k": k, "v": v, "a": a, "b": b}[what][70])[1] = float("inf")
    got = []
    for seg in (0, 1, 2):
        monkeypatch.setattr(ops, "_chunk_rule_seg", lambda *x, seg=seg: seg)
        s = st.clone()
        o = ops.gdn_scan(q, k, v, a, b, torch.zeros(H, device=DEV), torch.zeros(H, device=DEV), s, i32([0, T]), i32([0]), i32([0]), H, H)
        got.append((o.float(), s))
    for o, s in got[1:]:
        for x, y in ((o, got[0][0]), (s, got[0][1])):
            assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf())
            assert torch.allclose(x[y.isfinite()], y[y.isfinite()], rtol=2.0 ** -7, atol=1e-4)


@pytest.mark.parametrize("delta", [True, False])
def test_segments_are_as_exact_as_one_piece(delta, monkeypatch):
    """A long prompt of few heads, which the rule cuts, against 64 bits."""
    torch.manual_seed(11)
    T, H, dk, dv, errors = 1700, 2, 128, 64, []
    rule = ops._chunk_rule_seg
    assert rule(T, 1, H, dv, delta) > 0
    c, ab = torch.randn(T, 2 * H * dk + H * dv, device=DEV).to(BF), torch.randn(T, 2 * H, device=DEV).to(BF)
    q, k, v = c[:, :H * dk], c[:, H * dk:2 * H * dk], c[:, 2 * H * dk:]
    slow, sq = torch.linspace(-9, -6, H, device=DEV), (i32([0, T]), i32([0]), i32([0]))   # decays that a state outlives
    st, zero = torch.randn(1, H, dv, dk, device=DEV) * 0.2, torch.zeros(H, device=DEV)
    if delta:
        args, tail, scan, exact = (q, k, v, ab[:, :H], ab[:, H:], slow, zero), (H, H), ops.gdn_scan, exact_gdn
    else:
        args, tail, scan, exact = (v, ab[:, :H], k, q, -slow.exp(), zero, zero, 0.001), (H, dv, dk, H), ops.ssm_scan, exact_ssm
    want, want_state = exact(*args, st, *sq, *tail)
    for f in (lambda *a: 0, rule):
        monkeypatch.setattr(ops, "_chunk_rule_seg", f)
        s = st.clone()
        o = scan(*args, s, *sq, *tail)
        assert near(o, s, want, want_state)
        errors.append(((s.cpu().double() - want_state).norm() / want_state.norm()).item())
    print("state, one piece and segments:", errors)
    assert errors[1] <= 1.25 * errors[0]   # (another order of the same sums)


def test_silu_of_every_value():
    """The convolution's SiLU for all bf16 inputs, infinities and NaN among them: the value in 64 bits, rounded (one tap of 1, each
    row a sequence).  Where e^-x is past fp32 (x < -88.72) it is 0."""
    x = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(BF).view(256, 256).to(DEV)
    w = torch.zeros(256, 4, dtype=BF, device=DEV)
    w[:, 3] = 1
    y = ops.ssm_conv1d(x, w, None, torch.zeros(256, 256, 3, dtype=BF, device=DEV), i32(list(range(257))), i32(list(range(256))), i32([1] * 256))
    want = (x.double() / (1 + (-x.double()).exp())).to(BF)
    want[(x < -88.72) & x.isfinite()] = 0
    assert bool(((y == want) | (y.isnan() & want.isnan())).all())


@pytest.mark.parametrize("S", [2, 63, 64, 65])
@pytest.mark.parametrize("delta", [True, False])
def test_sequences_in_turn(S, delta):
    """Ragged sequences, equal ones and empty ones among them, on both sides of the number that is ordered by length, in a part of a round over
    the chip (few heads) and in many."""
    lens = [(0, 33, 1, 70, 3, 4, 33, 128)[(5 * i + i // 8) % 8] for i in range(S)]
    if delta:
        for dims in ((64, 16, 1, 5, 0), (64, 16, 2, 48, 0)):
            test_delta_rule_prompts(lens, *dims)
    else:
        for dims in ((3, 16, 64, 1, 0), (48, 16, 64, 2, 0)):
            test_selective_scan_prompts(lens, *dims)
