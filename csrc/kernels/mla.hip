// Multi-head latent attention (DeepSeek-V2/V3, Kimi-K2) in the absorbed
// form, for gfx950.
//
// Every layer caches one latent row per token: [c_kv (kv_lora_rank, kv_a_layernorm'd) | k_pe
// (roped)], paged as cache[pages, 16, DK] bf16 -- DK = 576 = 512 + 64 for DeepSeek-V2/V3 / Kimi-K2,
// 288 = 256 + 32 for MiniCPM3 (template instances below).  With W_UK folded into the query
// (q_lat = [q_nope . W_UK | q_pe], 576 wide) and W_UV applied after the attention, MLA is
// multi-QUERY attention over that latent: scores use all 576 dims, values are the first 512.
// Four kernels serve decode, prefill and chunked prefill: row tiles (mla_attn_rows_kernel, DK = 576: prompts, and
// decode steps of some 24 rows or 6 with many heads), 128 heads a workgroup (mla_attn_all_kernel: many decode rows of
// so many heads), and 16 heads a workgroup, of pages (mla_attn_pages_kernel, DK = 576: few rows) and here (other widths; a few rows over short tables): a work item is one query
// token x 16 heads (every head of a token shares the causal limit) x one split-K partition.
//
// Workgroup = 4 waves: all four compute S^T for the same 16 heads x 32 keys (the K tile is
// staged once in LDS and read by all), and each wave owns 128 of the 512 value dims.
//   S^T = K . Q^T     v_mfma_f32_16x16x32_bf16, A = K rows from LDS (ds_read_b128),
//                     B = Q held in registers (18 k-steps of 32 dims)
//   O^T += V^T . P^T  A = V^T from the SAME LDS image via ds_read_b64_tr_b16 (hardware
//                     transpose, cdna_hip_programming.md T10), B = P^T straight from the S^T
//                     accumulators in the permuted k-slot order of attention.hip
// LDS rows are 1152 B (72 x 16-B chunks); chunk x of key row r lives at x ^ (r & 7), which
// spreads both the row reads and the transposed reads over the banks.
#include "common.h"
#include "mma32.h"

#include <cstdlib>

#ifndef OME_NEG_INF
#define OME_NEG_INF (-__builtin_inff())
#endif

namespace {

constexpr int KT = 32;   // keys per iteration (two 16-token pages)
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16x32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// LDS row stride in 16-byte chunks, padded to a multiple of 8 so the xor swizzle stays in the row
template <int DK>
constexpr int lds_chunks() { return ((DK / 8) + 7) / 8 * 8; }
template <int DK>
__device__ __forceinline__ int swz(int row, int chunk) { return row * lds_chunks<DK>() + (chunk ^ (row & 7)); }

__device__ __forceinline__ bf16x4 tr_read(const bf16* lds_base, int byte_off) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (s16x4 __attribute__((address_space(3)))*)((__attribute__((address_space(3))) char*)(
          (__attribute__((address_space(3))) bf16*)lds_base) + byte_off));
  return __builtin_bit_cast(bf16x4, v);
}

// How many of `parts` partitions mla_attn_kernel cuts `tiles` key tiles into.  Beyond 16 a further one costs more to merge than it saves unless
// each keeps four tiles, so short contexts leave the later ones empty (one token of 16 heads, 16 / 32 / 64 partitions of equal size, us:
// 300 keys 11.6 / 13.0 / 15.8, 3000 23 / 21 / 24, 8000 44 / 31 / 31; every five or six tiles: 3000 23 / 23, 8000 31 / 31).
__device__ __forceinline__ int live_parts(int tiles, int parts) { return min(parts, max(16, (tiles + 3) / 4)); }
constexpr int LEAST_PAIRS = 2;   // key tiles of a partition of mla_attn_pages_kernel, whose waves take a page each

}  // namespace

template <int DK, int DV>
__global__ __launch_bounds__(256) void mla_attn_kernel(
    const bf16* __restrict__ q, int64_t q_stride_t, const bf16* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_row,
    const int* __restrict__ kv_lens, int H, float scale_log2, int parts, bf16* __restrict__ out,
    int64_t out_stride_t, float* __restrict__ ws_o, float* __restrict__ ws_ml, const float* __restrict__ sinks,
    int window) {
  constexpr int CH = DK / 8, NB = DV / 64, NST = (KT * CH + 255) / 256;   // NB 16-dim blocks per wave
  __shared__ __attribute__((aligned(16))) bf16 sK[KT * lds_chunks<DK>() * 8];
  const int t = blockIdx.x, h0 = blockIdx.y * 16, part = blockIdx.z;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = lane & 15, g = lane >> 4;
  const int L = kv_lens[t];
  const int lo = window > 0 ? max(L - window, 0) : 0;   // sliding window: keys [lo, L) only
  const int n_pages = (L + 15) >> 4;
  const int pairs = (n_pages + 1) >> 1;
  const int pair_lo = lo / KT;                          // key tiles wholly before the window are skipped
  const int live = live_parts(pairs - pair_lo, parts), per_part = (pairs - pair_lo + live - 1) / live;
  const int pair_begin = pair_lo + part * per_part, pair_end = min(pairs, pair_begin + per_part);
  const int* bt = block_tables + (int64_t)tok_row[t] * bt_stride;
  const int64_t ws_row = ((int64_t)t * H + h0 + col) * parts + part;

  const bool hv = h0 + col < H;   // head groups are 16 wide; the last may be partial (MiniCPM3: 40)

  // ---- Q^T operand: lane (col, g) holds Q[h0+col][32 s + 8 g + j] ----
  bf16x8 qf[DK / 32];
  const bf16* qp = q + (int64_t)t * q_stride_t + (int64_t)(hv ? h0 + col : 0) * DK + 8 * g;
#pragma unroll
  for (int s = 0; s < DK / 32; ++s) qf[s] = hv ? ld8(qp + 32 * s) : bf16x8{};

  f32x4 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = OME_NEG_INF, lsum = 0.f;

  // staging: 32 keys x CH chunks, NST per thread; chunk c -> (key c / CH, x c % CH)
  bf16x8 stage[NST];
  auto load_pair = [&](int pr) {
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = tid + 256 * i;
      if ((KT * CH) % 256 != 0 && c >= KT * CH) break;
      const int key = c / CH, x = c - key * CH;
      const int pg = 2 * pr + (key >> 4);
      const int page = bt[pg < n_pages ? pg : 0];
      stage[i] = ld8(cache + ((int64_t)page * 16 + (key & 15)) * DK + 8 * x);
    }
  };
  if (pair_begin < pair_end) load_pair(pair_begin);

  for (int pr = pair_begin; pr < pair_end; ++pr) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NST; ++i) {
      const int c = tid + 256 * i;
      if ((KT * CH) % 256 != 0 && c >= KT * CH) break;
      const int key = c / CH, x = c - key * CH;
      *reinterpret_cast<bf16x8*>(&sK[swz<DK>(key, x) * 8]) = stage[i];
    }
    __syncthreads();
    if (pr + 1 < pair_end) load_pair(pr + 1);

    // ---- S^T [32 keys x 16 heads] ----
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) {
      const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&sK[swz<DK>(col, 4 * s + g) * 8]);
      const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&sK[swz<DK>(16 + col, 4 * s + g) * 8]);
      s0 = mfma16x32(a0, qf[s], s0);
      s1 = mfma16x32(a1, qf[s], s1);
    }
    // ---- mask + online softmax (column = head, lane-local up to the 4 lane groups) ----
    const int kbase = pr * KT;
    float mx = OME_NEG_INF;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k0 = kbase + 4 * g + i, k1 = k0 + 16;
      s0[i] = (k0 < L && k0 >= lo) ? s0[i] * scale_log2 : OME_NEG_INF;
      s1[i] = (k1 < L && k1 >= lo) ? s1[i] * scale_log2 : OME_NEG_INF;
      mx = fmaxf(mx, fmaxf(s0[i], s1[i]));
    }
    mx = group4_max(mx);
    const float m_new = fmaxf(m, mx);
    const float alpha = (m_new == OME_NEG_INF) ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
    bf16x8 pb;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p0 = (m_new == OME_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(s0[i] - m_new);
      const float p1 = (m_new == OME_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(s1[i] - m_new);
      ps += p0 + p1;
      pb[i] = (bf16)p0;
      pb[4 + i] = (bf16)p1;
    }
    ps = group4_sum(ps);
    lsum = lsum * alpha + ps;
    m = m_new;
    // ---- O^T [this wave's DV / 4 dims x 16 heads] += V^T . P^T ----
    // tr-read block: rows = keys 4g + q (+16 for page B), cols = 16 dims; lane 4q+p of the
    // group addresses row q, columns 4p..4p+3.
    const int qrow = (lane & 15) >> 2, pcol = lane & 3;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int d0 = wave * (DV / 4) + 16 * nb + 4 * pcol;  // first of this lane's 4 dims
      const int ra = 4 * g + qrow, rb = 16 + 4 * g + qrow;
      const int oa = swz<DK>(ra, d0 >> 3) * 16 + (d0 & 7) * 2;
      const int ob = swz<DK>(rb, d0 >> 3) * 16 + (d0 & 7) * 2;
      const bf16x4 va = tr_read(sK, oa), vb = tr_read(sK, ob);
      bf16x8 a;
      a[0] = va[0]; a[1] = va[1]; a[2] = va[2]; a[3] = va[3];
      a[4] = vb[0]; a[5] = vb[1]; a[6] = vb[2]; a[7] = vb[3];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[nb][i] *= alpha;
      o[nb] = mfma16x32(a, pb, o[nb]);
    }
  }

  // ---- epilogue: O^T lane map dim = 16 nb + 4 g + i, head = col ----
  // sinks (optional, fp32 [H], natural-log units, unscaled): exp(sink_h) joins head h's softmax
  // denominator once, with no value; unsplit here, after the merge of the partials otherwise
  if (sinks != nullptr && parts == 1 && hv) {
    const float sk = sinks[h0 + col] * 1.4426950408889634f;
    const float m_fin = fmaxf(m, sk), a = __builtin_amdgcn_exp2f(m - m_fin);
    lsum = lsum * a + __builtin_amdgcn_exp2f(sk - m_fin);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[nb][i] *= a;
  }
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (!hv || (part >= 16 && pair_begin >= pair_end)) return;   // (of the partitions beyond 16 the merge reads none that is empty: 300 to 2500 keys 1.03 to 1.07 -> 1.01 to 1.03 of the time with 16)
  if (parts == 1) {
    bf16* op = out + (int64_t)t * out_stride_t + (int64_t)(h0 + col) * DV + wave * (DV / 4) + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(o[nb][i] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * nb) = v;
    }
  } else {
    float* wp = ws_o + ws_row * DV + wave * (DV / 4) + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      *reinterpret_cast<f32x4*>(wp + 16 * nb) = f32x4{o[nb][0] * inv, o[nb][1] * inv, o[nb][2] * inv,
                                                       o[nb][3] * inv};
    if (wave == 0 && g == 0) {
      ws_ml[2 * ws_row] = m;
      ws_ml[2 * ws_row + 1] = lsum;
    }
  }
}

// Sums of the lanes up to and with each (a row's lanes shifted, then the rows' last lanes broadcast), without LDS: a step of a __shfl is a round trip
__device__ __forceinline__ int wave_scan(int x) {
#define MLA_STEP(CTRL, ROWS) x += __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, true)
  MLA_STEP(0x111, 0xf);   // row_shr 1, 2, 4, 8
  MLA_STEP(0x112, 0xf);
  MLA_STEP(0x114, 0xf);
  MLA_STEP(0x118, 0xf);
  MLA_STEP(0x142, 0xa);   // row_bcast 15, 31
  MLA_STEP(0x143, 0xc);
#undef MLA_STEP
  return x;
}
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(wave_scan(x), 63); }
__device__ __forceinline__ int wave_most(int x) {   // the largest
#define MLA_STEP(CTRL, ROWS) x = max(x, __builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xf, false))
  MLA_STEP(0x111, 0xf);
  MLA_STEP(0x112, 0xf);
  MLA_STEP(0x114, 0xf);
  MLA_STEP(0x118, 0xf);
  MLA_STEP(0x142, 0xa);
  MLA_STEP(0x143, 0xc);
#undef MLA_STEP
  return __builtin_amdgcn_readlane(x, 63);
}

// A decode step's units (a token's tiles of heads, HG of them) in at most 256 pieces: workgroup w takes piece w.  The span is the smallest number of key tiles that cuts all units
// into at most 256 pieces: one a CU (also within each XCD, to which workgroups go in turn), and none longer
// than it has to be, however ragged the contexts.  Every wave finds it from the lengths: lane l holds
// tokens 4 l .. 4 l + 3.
// (unit, and its piece `part` of `my_parts`); false: there is none.
constexpr int SPAN = 2, UNITS = 256;
__device__ __forceinline__ bool decode_piece(const int* __restrict__ kv_lens, int T, int H, int HG, int parts, int& unit, int& part, int& my_parts) {
  const int lane = threadIdx.x & 63;
  int nt4[4], most = SPAN, all = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tk = 4 * lane + i;
    nt4[i] = tk < T ? (kv_lens[tk] + KT - 1) / KT : 0;
    most = max(most, nt4[i]);
    all += nt4[i];
  }
  auto count = [&](int span, int i) {   // (a quotient of tiles is off by one at most)
    const int n = nt4[i] + span - 1, about = (int)((float)n * __builtin_amdgcn_rcpf((float)span)), rest = n - about * span;
    return 4 * lane + i < T ? min(parts, max(1, about + (rest >= span) - (rest < 0))) : 0;
  };
  auto pieces = [&](int span) { return wave_total(count(span, 0) + count(span, 1) + count(span, 2) + count(span, 3)) * HG; };
  most = wave_most(most);
  all = wave_total(all) * HG;
  // all / span <= pieces <= all / span + units; one piece a unit is at most 256 (the caller's rule)
  int lo = max(SPAN, min(most, all / UNITS)), hi = T * HG < UNITS ? max(lo, min(most, all / (UNITS - T * HG) + 1)) : most;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pieces(mid) <= UNITS) hi = mid;
    else lo = mid + 1;
  }
  // pieces that save fewer key tiles than their partials' way to memory and back costs: none (64 heads, 128 rows of ~100
  // keys 34 -> 28 us)
  if (most - lo <= 2 + T * H / 2048) lo = most;
  const int w = blockIdx.x, c0 = count(lo, 0), c1 = count(lo, 1), c2 = count(lo, 2), c3 = count(lo, 3);
  const int incl = wave_scan(c0 + c1 + c2 + c3);
  if (w >= __builtin_amdgcn_readlane(incl, 63) * HG) return false;
  const int at = __popcll(__ballot(incl * HG <= w));            // the lane whose tokens piece w belongs to
  int tok = 4 * at, base = at ? __builtin_amdgcn_readlane(incl, at - 1) : 0;
  my_parts = __builtin_amdgcn_readlane(c0, at);
  if ((base + my_parts) * HG <= w) base += my_parts, ++tok, my_parts = __builtin_amdgcn_readlane(c1, at);
  if ((base + my_parts) * HG <= w) base += my_parts, ++tok, my_parts = __builtin_amdgcn_readlane(c2, at);
  if ((base + my_parts) * HG <= w) base += my_parts, ++tok, my_parts = __builtin_amdgcn_readlane(c3, at);
  const int hg = (w - base * HG) / my_parts;
  part = (w - base * HG) - hg * my_parts;
  unit = tok * HG + hg;
  return true;
}

// ------------------------------------------------------------------------------------------
// Few decode rows at DeepSeek's widths: work items and partitions of mla_attn_kernel, but each of the four waves streams pages of its own, every
// fourth of the partition's, with an online softmax of its own over all DV value dims, and the four meet in LDS at the end.  Bound by the
// cache's bytes where contexts are long, and by its latency where they are short: a wave has a page (18 KB) on its way to LDS while it multiplies
// another, 74 KB a CU, and no step waits for another wave.  (Above, 32 keys at a time go through registers, all waves form the same S^T, and
// two barriers a tile leave the loads of one tile of each workgroup in flight.)  Whole calls, us, that -> this: 16 heads, 8 rows of ~3000 and ~8000 keys
// 31 -> 27, 58 -> 38, 16 rows 43 -> 31, 85 -> 45, 23 rows of 400, 1000, 3000, 8000 22 -> 17, 32 -> 23, 67 -> 35, 138 -> 59; 32 heads, 12 rows of 1000 and 8000
// 31 -> 22, 156 -> 61; 64 heads, 4 of 3000 42 -> 29; 128 heads, 2 of 3000 34 -> 25; 8 heads, 40 of 1000 34 -> 24.  At 16 workgroups and fewer over
// 100 to 400 keys it took 0.2 to 1 us more (4 rows of 16 heads 11.7 -> 12.5, 14.0 -> 14.2; 1 of 128 over 92 pages 18.4 -> 18.9), so tables of at most 96 pages stay there.
// PLAN: decode steps of up to 16 heads that go to 32-row tiles, in their pieces by length; there half of a tile's rows are none, and one wave's products, 2 us
// a tile, are behind memory.  Them -> this, us: 128 rows of ~300, ~1000 and ~3000 keys 30 -> 27, 53 -> 44, 120 -> 105, 64 of 1000 33.6 -> 30.8, 32 of 8000 70 -> 60, 24
// of 3000 36 -> 35; short contexts of few rows not (24 of 400 17.1 -> 18.6, 48 of 150 16.2 -> 16.7): from 3000 pages of tables on.  32 heads as two units 116 -> 171 (100 of
// 4000), units' tiles dealt out in equal runs 101 -> 107.
// ------------------------------------------------------------------------------------------
template <int DK, int DV, bool PLAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mla_attn_pages_kernel(
    const bf16* __restrict__ q, int64_t q_stride_t, const bf16* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_row,
    const int* __restrict__ kv_lens, int T, int H, float scale_log2, int parts, int2* __restrict__ plan, bf16* __restrict__ out,
    int64_t out_stride_t, float* __restrict__ ws_o, float* __restrict__ ws_ml, const float* __restrict__ sinks,
    int window) {
  constexpr int CH = DK / 8, NV = DV / 16, NB = NV / 4, MOVES = 16 * CH / 64, IMG = 16 * CH * 16;
  static_assert(CH % 8 == 0 && MOVES * 64 == 16 * CH && 9 * 64 == 8 * CH, "whole moves, nine of them 8 rows");
  static_assert(NV * 1024 <= 2 * IMG, "a wave's output fits its images");
  __shared__ __attribute__((aligned(16))) char sK[4 * 2 * IMG];
  __shared__ float sM[4][16], sL[4][16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int HG = (H + 15) / 16;
  int unit = blockIdx.x, part = PLAN ? 0 : blockIdx.z;
  if (PLAN && parts > 1) {
    if (!decode_piece(kv_lens, T, H, HG, parts, unit, part, parts)) return;   // whole block
    if (part == 0 && tid == 0) plan[unit] = int2{(int)blockIdx.x, parts};
  }
  const int t = PLAN ? unit / HG : blockIdx.x, h0 = (PLAN ? unit - t * HG : (int)blockIdx.y) * 16;
  const int col = lane & 15, g = lane >> 4;
  const int L = __builtin_amdgcn_readfirstlane(kv_lens[t]);
  const int lo = window > 0 ? max(L - window, 0) : 0;   // sliding window: keys [lo, L) only
  const int n_pages = (L + 15) >> 4, pairs = (n_pages + 1) >> 1, pair_lo = lo / KT;   // partitions as in mla_attn_kernel
  const int live = PLAN ? parts : live_parts(pairs - pair_lo, parts), per_part = max(PLAN ? 0 : LEAST_PAIRS, (pairs - pair_lo + live - 1) / live);
  const int pair_begin = pair_lo + part * per_part, pair_end = min(pairs, pair_begin + per_part);
  const int p0 = 2 * pair_begin, p1 = min(2 * pair_end, n_pages);
  const int n = __builtin_amdgcn_readfirstlane(max(0, (p1 - p0 - wave + 3) >> 2));   // this wave's pages: p0 + wave, + 4, ..
  const int* bt = block_tables + (int64_t)tok_row[t] * bt_stride;
  const bool hv = h0 + col < H;
  const int64_t ws_row = PLAN ? (int64_t)blockIdx.x * 16 + col : ((int64_t)t * H + h0 + col) * parts + part;   // (PLAN: pieces' rows one after the other)
  bf16* const op = out + (int64_t)t * out_stride_t + (int64_t)(h0 + col) * DV + wave * (DV / 4) + 4 * g;
  if (p0 >= p1) {   // whole block: no keys (the merge reads no value of a partition whose sum is 0, and of those beyond 16 not the sum)
    if (hv && parts == 1) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) *reinterpret_cast<bf16x4*>(op + 16 * nb) = bf16x4{};
    } else if (hv && (PLAN || part < 16) && wave == 0 && g == 0) {
      ws_ml[2 * ws_row] = OME_NEG_INF;
      ws_ml[2 * ws_row + 1] = 0.f;
    }
    return;
  }

  // The first two pages by scalar loads: their moves wait for neither the queries nor the list
  const int first = bt[min(p0 + wave, p1 - 1)], second = bt[min(p0 + wave + 4, p1 - 1)];
  const auto id = [&](int i) { const int p = p0 + wave + 4 * (i + lane); return bt + (p < p1 ? p : p0); };
  int pages = *id(0), at0 = 0;   // the next 64 of this wave's pages, one a lane
  // ---- Q^T operand: lane (col, g) holds Q[h0+col][32 s + 8 g + j] ----
  bf16x8 qf[DK / 32];
  const bf16* qp = q + (int64_t)t * q_stride_t + (int64_t)(hv ? h0 + col : 0) * DK + 8 * g;
#pragma unroll
  for (int s = 0; s < DK / 32; ++s) qf[s] = hv ? ld8(qp + 32 * s) : bf16x8{};

  // A page -> LDS image: move i writes chunks [64 i, 64 i + 64), each lane fetching the source chunk that its row's swizzle puts there
  uint32_t ofs[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    const int c = 64 * j + lane, r = c / CH;
    ofs[j] = (r * CH + ((c - r * CH) ^ (r & 7))) * 16;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sK + wave * 2 * IMG;
  const auto look = [&](int i) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)   // (waited for here: the compiler would wait at every use, and for the moves as well)
    asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=&v"(pages) : "v"(id(i)) : "memory");
#endif
    at0 = i;
  };
  const auto move_page = [&](int i, int index) __attribute__((always_inline)) {
    const bf16* page = cache + (int64_t)index * 16 * DK;
    const uint32_t bytes = min(16, L - 16 * (p0 + wave + 4 * i)) * DK * 2;   // (rows past the context: zeros)
#pragma unroll
    for (int j = 0; j < MOVES; ++j) buffer_to_lds(page, bytes, ofs[j % 9] + j / 9 * (8 * CH * 16), 0, lds0 + (i & 1) * IMG + 1024 * j);
  };
  const auto move = [&](int i) __attribute__((always_inline)) {
    if (i >= n) return;
    if (i - at0 == 64) look(i);
    move_page(i, __builtin_amdgcn_readlane(pages, i - at0));
  };
  f32x4 o[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = OME_NEG_INF, lsum = 0.f;
  if (n > 0) move_page(0, first);
  if (n > 1) move_page(1, second);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int s = 0; s < DK / 32; ++s) asm volatile("" : "+v"(qf[s]));   // (waited for here, once)
  asm volatile("" : "+v"(pages));
#endif
  const int qrow = col >> 2, pcol = lane & 3, row = 4 * g + qrow;   // tr-read block: rows = keys 4 g + qrow, columns 4 pcol .. + 3
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    if (i + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MOVES) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const bf16* img = reinterpret_cast<const bf16*>(sK + (wave * 2 + (i & 1)) * IMG);
    // ---- S^T [16 keys x 16 heads], two chains ----
    f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) sc[s & 1] = mfma16x32(*reinterpret_cast<const bf16x8*>(&img[swz<DK>(col, 4 * s + g) * 8]), qf[s], sc[s & 1]);
    const int k0 = 16 * (p0 + wave + 4 * i) + 4 * g;
    f32x4 s = sc[0] + sc[1];
    float mx = OME_NEG_INF;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = (k0 + e < L && k0 + e >= lo) ? s[e] * scale_log2 : OME_NEG_INF;
      mx = fmaxf(mx, s[e]);
    }
    mx = group4_max(mx);
    const float m_new = fmaxf(m, mx);
    const float alpha = m_new == OME_NEG_INF ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
    // Weights as they are used: their rounding cancels in the quotient.  PLAN: with what rounding took from them in a second product, as the row tiles have it of
    // weights that stand out (3% of the time; error against 64 bits 0.0017 instead of 0.0018, theirs 0.0017 to 0.0018)
    s16x4 pb, pr;
    float ps = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float p = m_new == OME_NEG_INF ? 0.f : __builtin_amdgcn_exp2f(s[e] - m_new);
      const bf16 high = (bf16)p;
      ps += PLAN ? p : (float)high;
      pb[e] = __builtin_bit_cast(short, high);
      pr[e] = __builtin_bit_cast(short, (bf16)(p - (float)high));
    }
    lsum = lsum * alpha + group4_sum(ps);
    m = m_new;
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int v = 0; v < NV; ++v) o[v] *= alpha;
    }
    // ---- O^T [DV x 16 heads] += V^T . P^T ----
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const s16x4 val = __builtin_bit_cast(s16x4, tr_read(img, swz<DK>(row, 2 * v + (pcol >> 1)) * 16 + (pcol & 1) * 8));
      if constexpr (PLAN) o[v] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(val, pr, o[v], 0, 0, 0);
      o[v] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(val, pb, o[v], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the image is read)
    move(i + 2);
  }

  // ---- the waves' sums meet: each writes its own over its images, and takes a quarter of the dims of all ----
  f32x4* const so = reinterpret_cast<f32x4*>(sK);
  constexpr int WO = 2 * IMG / 16;   // between waves
#pragma unroll
  for (int v = 0; v < NV; ++v)
    if (n > 0) so[wave * WO + v * 64 + lane] = o[v];
  if (g == 0) sM[wave][col] = m, sL[wave][col] = lsum;
  __syncthreads();
  const int act = min(4, p1 - p0);   // waves that had a page
  f32x4 sum[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) sum[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  m = OME_NEG_INF, lsum = 0.f;
  for (int w = 0; w < act; ++w) m = fmaxf(m, sM[w][col]);
  for (int w = 0; w < act; ++w) {
    const float mw = sM[w][col], e = mw == OME_NEG_INF ? 0.f : __builtin_amdgcn_exp2f(mw - m);
    lsum += e * sL[w][col];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sum[nb] += e * so[w * WO + (wave * NB + nb) * 64 + lane];
  }

  // ---- output or partials: dim = 16 nb + 4 g + i of the wave's quarter, head = col ----
  if (!PLAN && sinks != nullptr && parts == 1 && hv) {
    const float sk = sinks[h0 + col] * 1.4426950408889634f;
    const float m_fin = fmaxf(m, sk), a = __builtin_amdgcn_exp2f(m - m_fin);
    lsum = lsum * a + __builtin_amdgcn_exp2f(sk - m_fin);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sum[nb] *= a;
  }
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (!hv) return;
  if (parts == 1) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(sum[nb][i] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * nb) = v;
    }
  } else {
    float* wp = ws_o + ws_row * DV + wave * (DV / 4) + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) *reinterpret_cast<f32x4*>(wp + 16 * nb) = sum[nb] * inv;
    if (wave == 0 && g == 0) {
      ws_ml[2 * ws_row] = m;
      ws_ml[2 * ws_row + 1] = lsum;
    }
  }
}

// ------------------------------------------------------------------------------------------
// Row tiles: one workgroup of NW waves owns 32 * NW neighbouring query rows (row = token * H + head) and one
// split-K partition, so that each latent key tile is streamed and staged in LDS ONCE for all of them: the heads
// of one token in decode, the heads of several prompt tokens of a sequence otherwise (the 16-head
// kernel above streams the prefix again for every token, and its four waves each compute the same S^T).  A workgroup
// takes the tokens of one block-table row only: the tile's own the first, one more for each sequence that begins inside
// a tile.  The others' rows ride along with weights 0 and are not stored (0 times an infinite or NaN value of a
// broken sequence is NaN, which must stay in that sequence).
//
// Bound by the matrix cores, with LDS reads close behind: a wave owns 32 rows and all DV value dims, so each
// LDS operand feeds 32 columns (16 rows a wave, the layout before, read every key tile eight times per
// 128 rows).  That takes one wave per SIMD: O^T [DV x 32] fills the 256 accumulation registers, Q^T 144 of
// the others.
//   S^T [32 keys x 32 rows] = K . Q^T   (DK/16 MFMAs 32x32x16, lane = key / row, 8 dims a lane half)
//   O^T [DV x 32] += V^T . P^T          (DV/32 x 2 MFMAs; V^T by hardware-transposed LDS reads, key order of S^T)
// Nothing else runs on the SIMD meanwhile, so the loop is pipelined by hand.  A product takes 32 cycles of the matrix cores and 4 of issue, so up
// to six vector instructions beside it cost next to nothing: the softmax of tile n stands between the products of S^T of tile n + 1 (the
// exponentials of its last 16 keys between those of O^T), and of 128 rows the nine moves of tile n + 3 one by one beside the last products of O^T (four
// images; nine in a row hold a wave up for some 450 cycles).  A branch beside each product, taken or not, costs 40 cycles, so the loop
// has none there.  Of 128 rows, 256 workgroups of 100 tiles that share their keys, a tile took 2.65 us with moves and softmax ahead of the products and
// takes 2.42; its products alone take 1.65, the rate at which the card runs out of power (1380 TFLOP/s): the rest is LDS reads at 128 bytes a
// cycle, which the products need all of, and waiting for the wave whose weights stand out most often.
// O^T is rescaled only where a row's maximum rose by more than 2^8 since its last rescale (weights stay below
// 2^8), almost never after a row's first tile.  A row's largest weight is then not exactly 1, as in the 16-head
// kernel, so its rounding to bf16 counts: the keys with a weight that stands out are multiplied a second time with what
// rounding took (16 keys of all rows at once; w^2 over 16, or of decode steps 6, times the mean of the squares of the
// largest weight of each tile so far, or any that may come to a row's largest where there are fewer tiles than that).
// The denominator sums the weights as they are used.  Error against 64 bits over the shapes of DeepSeek's heads
// 0.0017..0.0018 of the result (16-head kernel 0.0017..0.0019; without the second product 0.0019..0.0021, in 0.87 of the
// time).
//
// Measured (16-head kernel, or for decode the 16-row waves before -> now): three prompts of 3394 rows x 16 heads
// 738 -> 135 us (118 -> 645 TFLOP/s); decode, 48 contexts of ~3000 keys x 128 heads 100 -> 86 us.
// ------------------------------------------------------------------------------------------
// The products (mma32.h): with one wave per SIMD, what covers an LDS read is the distance to its product.  `mma_new` comes after a
// VALU write of its operands.
__device__ __forceinline__ void mma_new(f32x16& c, bf16x8 a, bf16x8 b) {   // c = a b
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 3\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b) : "memory");
#endif
}
__device__ __forceinline__ void mma_last(f32x16& d, bf16x8 a, bf16x8 b, const f32x16& c) {   // d = c + a b, which others may read
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3\n\t" MMA_WAIT : "=&v"(d) : "v"(a), "v"(b), "v"(c) : "memory");
#endif
}
// Chunk x of key row r lies at x ^ row_swz(r): the same chunk of 16 rows, and four chunks of four, in all of the 64 banks (rows are 9 times
// half of them wide)
__device__ __forceinline__ int row_swz(int r) { return (r >> 1 & 1) << 2 | (r >> 2 & 1) << 1 | (r >> 3 & 1); }

// First token whose block-table row is e, by a 64-way search of the whole wave; -1: none.  tok_row ascends in the
// runtime's prompts; of rows in any other order it may miss e, the same way for every caller.
__device__ __forceinline__ int first_token(const int* __restrict__ tok_row, int T, int e) {
  const int lane = threadIdx.x & 63;
  int lo = 0, n = T;   // it is in [lo, lo + n]
  while (n > 0) {
    const int step = (n + 63) >> 6, d = lane * step;
    const uint64_t rest = __ballot(d >= n || tok_row[lo + d] >= e);
    const int k = rest ? __builtin_ctzll(rest) : 64;   // tokens before lane k's are below e
    if (k == 0) break;
    const int at = (k - 1) * step + 1;
    n = min(k * step, n) - at;
    lo += at;
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  return lo < T && tok_row[lo] == e ? lo : -1;
}

// One query row over L keys by one wave, lane = key, then 8 value dims: to `out`, or as a partial in the row tiles' layout
template <int DK, int DV>
__device__ __forceinline__ void plain_row(const bf16* q, const bf16* cache, const int* bt, int L, float scale_log2, bool whole,
                                          bf16* out, float* part_o, float* part_ml) {
  const int lane = threadIdx.x & 63;
  float m = OME_NEG_INF, l = 0.f, acc[8] = {};
  for (int k0 = 0; k0 < L; k0 += 64) {
    const int key = min(k0 + lane, L - 1);
    const bf16* kv = cache + ((int64_t)bt[key >> 4] * 16 + (key & 15)) * DK;
    float s = 0.f;
#pragma unroll 1
    for (int c = 0; c < DK; c += 8) {
      const bf16x8 a = ld8(q + c), b = ld8(kv + c);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += (float)a[e] * (float)b[e];
    }
    s = k0 + lane < L ? s * scale_log2 : OME_NEG_INF;
    float mn = fmaxf(m, s);
    for (int x = 32; x > 0; x >>= 1) mn = fmaxf(mn, __shfl_xor(mn, x));
    const float alpha = m == OME_NEG_INF ? 0.f : __builtin_amdgcn_exp2f(m - mn);
    const float p = mn == OME_NEG_INF ? 0.f : __builtin_amdgcn_exp2f(s - mn);
    float ps = p;
    for (int x = 32; x > 0; x >>= 1) ps += __shfl_xor(ps, x);
    l = l * alpha + ps;
    m = mn;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll 1
    for (int j = 0; j < min(64, L - k0); ++j) {
      const float w = __shfl(p, j);
      const bf16x8 v = ld8(cache + ((int64_t)bt[(k0 + j) >> 4] * 16 + ((k0 + j) & 15)) * DK + 8 * lane);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += w * (float)v[e];
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  static_assert(DV == 512, "8 dims a lane");
  if (whole) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)(acc[e] * inv);
    st8(out + 8 * lane, o);
  } else {   // dims 8 lane .. + 3 belong to the tile's lane (row, half 0), the next four to (row, half 1)
    *reinterpret_cast<f32x4*>(part_o + lane * 256) = f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    *reinterpret_cast<f32x4*>(part_o + lane * 256 + 128) = f32x4{acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv};
    if (lane == 0) part_ml[0] = m, part_ml[1] = l;
  }
}

// Waves beside the NW that multiply which move the keys to LDS: one on each SIMD that has none.  A move holds its wave up for some 50 cycles, and the 36
// of a tile by the one wave of 32 rows took as long as its products.  Whole calls, us, moved by the waves that multiply -> by others: 32 rows,
// 16 heads, 24 x 3000 keys 40.5 -> 35.9, 32 x 8000 83 -> 70, 128 x 3000 145 -> 120; 64 rows, 64 heads, 48 x 3000 63.7 -> 60.4, 100 x 1500 74 -> 69.6;
// 100 prompt rows of 16 heads over 2000 keys 40.8 -> 38.7.  (128 rows have a wave on every SIMD, each with all of its registers.)
constexpr int row_movers(int NW) { return 4 - NW; }

template <int DK, int DV, int NW, bool DECODE>
__global__ __launch_bounds__(64 * (NW + row_movers(NW))) __attribute__((amdgpu_waves_per_eu(1, 1))) void mla_attn_rows_kernel(
    const bf16* __restrict__ q, int64_t q_stride_t, const bf16* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_row,
    const int* __restrict__ kv_lens, int T, int H, int seqs, float scale_log2, int parts, int2* __restrict__ plan,
    bf16* __restrict__ out, int64_t out_stride_t, float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  static_assert(DK == 576 && lds_chunks<DK>() == DK / 8, "LDS DMA image assumes unpadded 72-chunk rows");
  constexpr int MW = row_movers(NW), ML = MW ? MW : NW;   // ML waves move
  constexpr int CH = DK / 8, NI = KT * CH / 64, NJ = NI / ML, NV = DV / 32, NS = DK / 16;
  static_assert(NI % ML == 0 && (MW == 0 || NI / 2 % MW == 0), "whole DMA instructions per wave");
  constexpr int IMG = KT * CH * 16;   // bytes per key-tile image
  constexpr float LAZY = 8.f;
  constexpr int AHEAD = 4;            // LDS operands in flight: 4 x 32 cycles of matrix work cover a read
  __shared__ __attribute__((aligned(16))) char sK[4 * IMG];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sK;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  constexpr int RT = 32 * NW;
  // DECODE: a tile is RT heads of one token, and contexts are cut by length; else RT rows of [T * H], and the
  // workgroups past the tiles (`own_seq`) take a sequence's first rows where it begins inside a tile
  const int R = T * H, HG = (H + RT - 1) / RT;
  int unit = DECODE ? blockIdx.x : gridDim.x - 1 - blockIdx.x, part = blockIdx.y, my_parts = parts;   // (longest rows first)
  int own_seq = 0, own_first = 0;
  if constexpr (!DECODE) {
    own_seq = max(unit - (R + RT - 1) / RT + 1, 0);
    if (own_seq > 0) {
      own_first = first_token(tok_row, T, own_seq);
      if (own_first < 0) return;   // whole block
      unit = (int)((int64_t)own_first * H / RT);
    }
  }
  if (DECODE && parts > 1) {
    if (!decode_piece(kv_lens, T, H, HG, parts, unit, part, my_parts)) return;   // whole block
    if (part == 0 && tid == 0) plan[unit] = int2{(int)blockIdx.x, my_parts};
  }
  const int row0 = DECODE ? unit / HG * H + unit % HG * RT : unit * RT;
  const int row_end = DECODE ? (unit / HG + 1) * H : R;
  // the tile's tokens (at most 64: H >= 4), one a lane; the same in every wave
  const int t0 = row0 / H, nt = (min(row0 + RT, row_end) - 1) / H - t0 + 1;
  const int tl_row = tok_row[t0 + min(lane, nt - 1)], tl_len = kv_lens[t0 + min(lane, nt - 1)];
  uint64_t left = nt >= 64 ? ~0ull : (1ull << nt) - 1;
  if (own_seq > 0) {
    const uint64_t theirs = left & __ballot(tl_row == own_seq);
    if (own_first == t0 || own_first != t0 + __builtin_ctzll(theirs)) return;   // the tile's own workgroup takes them
    left = theirs;
  }
  // One pass: block-table row `bt_row`, whose tokens `same` marks
  const auto walk = [&](int bt_row, bool same, int lane) __attribute__((always_inline)) {
    const int col = lane & 31, hf = lane >> 5;
    const int row = row0 + wave * 32 + col;                           // this lane's row (S^T / O^T column)
    const bool hv = row < row_end;
    const int t = min(DECODE ? unit / HG : row / H, T - 1), head = hv ? row - t * H : 0;
    const int my_row = tok_row[t], my_len = hv ? kv_lens[t] : 0;
    // LDS lane bases; the XOR swizzle acts on the low three bits of a chunk index, the rest are immediates.
    // S^T reads chunk 2 s + hf of key row col; V^T reads, for 16-lane group gr = lane / 16, rows 4 hf + qr (+ 8, 16, 24)
    // and chunk 4 v + 2 (gr & 1) + pc / 2.
    const int gr = lane >> 4, qr = (lane & 15) >> 2, pc = lane & 3;
    uint32_t sofs[4], vofs[2], vofs8[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) sofs[e] = (col * CH + ((2 * e + hf) ^ row_swz(col))) * 16;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      vofs[e] = ((4 * hf + qr) * CH + ((4 * e + 2 * (gr & 1) + (pc >> 1)) ^ row_swz(4 * hf + qr))) * 16 + (pc & 1) * 8;
      vofs8[e] = (vofs[e] ^ 16) + 8 * CH * 16;   // of the row 8 further on
    }
    auto kfrag = [&](uint32_t img, int s) { return *reinterpret_cast<const bf16x8*>(sK + (sofs[s & 3] + img) + (s >> 2) * 128); };
    // The queries: a wave's 32 rows are one image, so they come as a tile of keys does, 1 KB a move, and out of LDS into registers.  (Straight into
    // registers a lane holds 16 bytes of its row at a time, 32 rows of two lanes: 128 rows 5.7 us on every CU at once, now 4.2; fewer rows are no slower so.)
    bf16x8 qf[NS];
    const bool moved = MW == 0 && (((uintptr_t)q | (uintptr_t)(2 * q_stride_t)) & 15) == 0 && (uint64_t)q_stride_t < 1 << 26;   // (9 tokens a wave: 32-bit offsets)
    if (moved) {
      const int tw = __builtin_amdgcn_readfirstlane(t);
      const uint32_t at = 2 * ((uint32_t)(t - tw) * (uint32_t)q_stride_t + (uint32_t)head * DK);
#pragma unroll
      for (int b = 0; b < 9; ++b) {
        const int c = 64 * b + lane, r8 = c / CH, x = (c - r8 * CH) ^ row_swz(r8);
#pragma unroll
        for (int a = 0; a < 4; ++a)
          buffer_to_lds(q + (int64_t)tw * q_stride_t, 0x7fffffffu, (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (8 * a + r8), (int)at) + 16 * (x ^ (a & 1)), 0,
                        lds0 + wave * IMG + 1024 * (9 * a + b));
      }
    } else if (MW == 0 || wave < NW) {
      const bf16* qp = q + (int64_t)t * q_stride_t + (int64_t)head * DK + 8 * hf;
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] = ld8(qp + 16 * s);
    }
    const int Lmax = wave_most(same ? tl_len : 0);
    const int* bt = block_tables + (int64_t)bt_row * bt_stride;
    const int n_pages = (Lmax + 15) >> 4, tiles = (n_pages + 1) >> 1, per = (tiles + my_parts - 1) / my_parts;
    const int begin = part * per, end = min(tiles, begin + per);
    // Key tile -> LDS image: instruction i writes chunks [64 i, 64 i + 64) lane-linearly, each lane fetching the source
    // chunk that the row's XOR swizzle puts there.  A page is 16 rows x 72 chunks = 18 instructions, so each
    // instruction reads one page: its descriptor is based at that page.
    // Nine instructions are 8 rows; those of the next 8 differ in the chunk's lowest bit (row_swz).
    static_assert(9 * 64 == 8 * CH && NI == 36, "9 offsets a lane");
    const int mv = MW ? wave - NW : wave;   // (of a wave that moves)
    uint32_t dofs2[5] = {};   // two in a register (below 2^15)
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int c = 64 * ((mv + ML * j) % (NI / 2)) + lane, kr = c / CH;
      dofs2[j >> 1] |= (uint32_t)((kr * CH + ((c - kr * CH) ^ row_swz(kr))) * 16) << 16 * (j & 1);
    }
    // The pages of 32 tiles from `pg0` on, one a lane: a scalar load on its way would turn every wait for an LDS operand
    // into one for all of them.
    int pages = 0, pg0 = 0;
    auto look = [&](int tile) {
      const int p = 2 * tile + lane;
#if defined(__HIP_DEVICE_COMPILE__)   // (waited for here: the compiler would wait before every use, and for the moves as well)
      asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=&v"(pages) : "v"(begin < end ? bt + (p < n_pages ? p : 0) : tok_row) : "memory");
#endif
      pg0 = tile;
    };
    // (The queries have come by then too.  The compiler, which does not know the moves, would otherwise wait for a query ahead of every product of S^T,
    // in the loop too, and so for all but a few of the moves that come after it.)
    if (MW == 0 || wave >= NW) look(begin);
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (moved) {
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] = kfrag(wave * IMG, s);
    }
#if defined(__HIP_DEVICE_COMPILE__)
    if (MW == 0 || wave < NW) {
#pragma unroll
      for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(qf[s]));
    }
#endif
    if constexpr (MW == 0) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __syncthreads();   // (the images are the keys' from here on)
    }
    int first_page = 0, second_page = 0;   // of the tile on its way (their addresses are formed beside the products, where they cost nothing), its image, its descriptors' size
    uint32_t to = 0, bytes = 0;
    auto aim = [&](int tile, int img) {    // (of a tile past the last nothing is read, zeros are written)
      if (tile < end && tile - pg0 == 32) look(tile);
      const int at = 2 * (tile - pg0);
      first_page = __builtin_amdgcn_readlane(pages, at & 63);
      second_page = __builtin_amdgcn_readlane(pages, (at + 1) & 63);
#if defined(__HIP_DEVICE_COMPILE__)
      if constexpr (MW == 0) asm volatile("" : "+s"(first_page), "+s"(second_page));
#endif
      to = lds0 + img * IMG + 64 * 16 * mv;
      bytes = tile < end ? 16 * DK * 2 : 0;
      asm volatile("" : "+v"(dofs2[0]), "+v"(dofs2[1]), "+v"(dofs2[2]), "+v"(dofs2[3]), "+v"(dofs2[4]));   // (or the loop would hold them unpacked)
    };
    auto landed = [&](bool more) {   // the tile before the one that was moved last (`more`: if one was)
      if (MW == 0 || more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NJ) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    auto dma = [&](int j) __attribute__((always_inline)) {
      const int i = mv + ML * j;
      constexpr int OWN = MW ? NI / 2 / ML : 9;   // offsets that a lane has: of a page's moves (MW == 0: two pages have an odd number)
      const uint32_t two = dofs2[j % OWN >> 1], at = j % OWN & 1 ? two >> 16 : two & 0xffff;
      const int page = j < NJ / 2 || (NJ % 2 && j == NJ / 2 && i < NI / 2) ? first_page : second_page;
      buffer_to_lds(cache + (int64_t)page * 16 * DK, bytes, at, 0, to + 64 * 16 * ML * j);
    };
    if constexpr (MW > 0) {
      if (wave >= NW) {   // three tiles ahead of the one whose values are multiplied; barriers as below
        const auto put = [&](int tile, int img) __attribute__((always_inline)) {
          if (tile >= end) return;
          aim(tile, img);
#pragma unroll
          for (int j = 0; j < NJ; ++j) dma(j);
        };
        if (begin < end) {
          put(begin, 0);
          put(begin + 1, 1);
          landed(begin + 1 < end);
          __syncthreads();
          put(begin + 2, 2);
          landed(begin + 2 < end);
          __syncthreads();
          for (int n = begin; n < end; ++n) {
            put(n + 3, (n + 3 - begin) & 3);
            landed(n + 3 < end);
            __syncthreads();
          }
        }
        __syncthreads();
        return;
      }
    }

    f32x16 o[NV];

    auto score = [&](uint32_t img, f32x16& to, auto&& beside) __attribute__((always_inline)) {   // S^T of the tile in image `img` (byte offset)
      f32x16 a;
      bf16x8 k[AHEAD];   // operands on their way from LDS
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) k[s] = kfrag(img, s);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (s == 0) mma_new(a, k[0], qf[0]);
        else if (s + 1 < NS) mma_add(a, k[s % AHEAD], qf[s]);
        else mma_last(to, k[s % AHEAD], qf[s], a);
        if (s + AHEAD < NS) k[s % AHEAD] = kfrag(img, s + AHEAD);
        beside(s);
        __builtin_amdgcn_sched_barrier(0);   // what stands beside a product stays there
      }
    };
    auto vfrag = [&](uint32_t img, int v, int st) {
      const int add = (v >> 1) * 128 + st * 16 * CH * 16;
      const bf16x4 x = tr_read(reinterpret_cast<const bf16*>(sK), vofs[v & 1] + img + add), y = tr_read(reinterpret_cast<const bf16*>(sK), vofs8[v & 1] + img + add);
      return bf16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    };

    const bool mine = hv && my_row == bt_row;
    const int L = mine ? my_len : 0;
    float m = OME_NEG_INF, lsum = 0.f;
    // the squares of the largest weight of each tile, summed: what a weight's error is measured against
    float peaks = 0.f, walked = 0.f;
    const float large = min((end - begin) * my_parts, DECODE ? 6 : 16);
    f32x16 sc;
    // The first two tiles together, the third beside the first one's products: the second was asked for beside them as well, and pieces of two
    // and three tiles, which saw its whole latency, took as much longer as the pipeline saved (us, three images -> that -> this: 16 rows of 128
    // heads over 640 keys 30.4 -> 30.5 -> 30.2, six prompts of 59 rows 36.9 -> 37.5 -> 36.4; 32 x 8000 keys of 16 heads 84.8 -> 85.9 -> 84.0).
    if (MW == 0 && begin < end) {
      aim(begin, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) dma(j);
      aim(begin + 1, 1);
#pragma unroll
      for (int j = 0; j < NJ; ++j) dma(j);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[v][i] = 0.f;
    if (begin < end) {
      if (MW == 0) landed(true);
      __syncthreads();
      static_assert(MW > 0 || NS % NJ == 0, "a move every so many products");
      score(0, sc, [&](int s) __attribute__((always_inline)) {
        if (MW == 0 && s == 0) aim(begin + 2, 2);
        if (MW == 0 && s % (NS / NJ) == 0) dma(s / (NS / NJ));
      });
      if (MW == 0) landed(true);
      __syncthreads();
    }
    const int Lmin = -wave_most(-L);   // the wave's shortest row: tiles below it have no key to mask
    int cur = 0;
    for (int n = begin; n < end; ++n) {
      const int nxt = (cur + 1) & 3;
      if (MW == 0) aim(n + 3, (cur + 3) & 3);   // (that image was last read in the previous round, before its barrier)
      if ((n + 1) * KT > Lmin) {
        const int key = n * KT + 4 * hf;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = key + 8 * (i >> 2) + (i & 3) < L ? sc[i] : OME_NEG_INF;
      }
      // The softmax, in pieces that stand beside the products of the next tile's scores: up to six vector instructions beside each cost
      // next to nothing.
      float ma = OME_NEG_INF, mb = OME_NEG_INF;   // of the lane's keys of the first and second 16, unscaled
      float mx, mn, ms, wt, ps = 0.f;             // ps: of the weights as they are used: their rounding cancels in the quotient
      bool rise;
      uint64_t two[2];
      float p[16];
      bf16x8 pb[2];
      const auto piece = [&](int s) __attribute__((always_inline)) {
        if (s < 8) {
          if (s < 4) ma = fmaxf(ma, fmaxf(sc[2 * s], sc[2 * s + 1]));
          else mb = fmaxf(mb, fmaxf(sc[2 * s], sc[2 * s + 1]));
        } else if (s == 8) {
          mx = fmaxf(ma, mb);
          auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
          mx = vmax_f32(__uint_as_float(w[0]), __uint_as_float(w[1])) * scale_log2;
        } else if (s == 9) {
          rise = mx > m + LAZY;   // (also a row's first tile: m = -inf)
          mn = rise ? mx : m;
          ms = mn == OME_NEG_INF ? 0.f : mn;
        } else if (s == 10) {
          // keys of this half or that among which a row has a weight that stands out: used in two parts
          const float wa = __builtin_amdgcn_exp2f(ma * scale_log2 - ms), wb = __builtin_amdgcn_exp2f(mb * scale_log2 - ms);
          const float far = large * peaks;
          two[0] = __ballot(!rise && wa * wa * walked > far);
          two[1] = __ballot(!rise && wb * wb * walked > far);
        } else if (s == 11) {
          wt = __builtin_amdgcn_exp2f(mx - ms);
        }
      };
      const auto weights = [&](int i, int part) __attribute__((always_inline)) {   // of keys i and i + 1, in four pieces
        if (part == 0) {
          if (i < 8) p[i] = sc[i] * scale_log2 - ms, p[i + 1] = sc[i + 1] * scale_log2 - ms;
          p[i] = __builtin_amdgcn_exp2f(p[i]);
        } else if (part == 1) {
          p[i + 1] = __builtin_amdgcn_exp2f(p[i + 1]);
        } else if (part == 2) {
          const bf16x2 h = {(bf16)p[i], (bf16)p[i + 1]};
          pb[i >> 3][i & 7] = h[0];
          pb[i >> 3][(i & 7) + 1] = h[1];
        } else {
          ps += (float)pb[i >> 3][i & 7] + (float)pb[i >> 3][(i & 7) + 1];
        }
      };
      if (n + 1 < end) {
        score(nxt * IMG, sc, [&](int s) __attribute__((always_inline)) {
          piece(s);
          if (s >= 12 && (s - 12) % 6 < 4) weights((s - 12) / 6 * 2, (s - 12) % 6);   // (the first half's)
          if (s >= 12 && s < 20) p[s - 4] = sc[s - 4] * scale_log2 - ms;   // (the second half's follow beside O's products)
        });
      } else {
#pragma unroll
        for (int s = 0; s < 12; ++s) piece(s);
#pragma unroll
        for (int i = 0; i < 8; i += 2)
#pragma unroll
          for (int part = 0; part < 4; ++part) weights(i, part);
#pragma unroll
        for (int i = 8; i < 16; ++i) p[i] = sc[i] * scale_log2 - ms;
      }
      bf16x8 vf[AHEAD];
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) vf[k] = vfrag(cur * IMG, k, 0);
      if (__ballot(rise && m != OME_NEG_INF)) {   // (a first tile has nothing to rescale: O^T and the sum are zero)
        const float alpha = rise && m != OME_NEG_INF ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
        lsum *= alpha;
        peaks *= alpha * alpha;
        // in the accumulation registers, by asm: as plain C++ all 256 products are computed every time and moved
        // through the other registers.  (waits: the last MFMA's results; the next one's operands)
        asm volatile(MMA_WAIT ::: "memory");
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float x = o[v][i];
#if defined(__HIP_DEVICE_COMPILE__)   // ("a": an accumulation register, unknown to the host pass)
            float y;
            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                         : "+a"(x), "=&v"(y)
                         : "v"(alpha));
#endif
            o[v][i] = x;
          }
        asm volatile("s_nop 7" ::: "memory");
      }
      peaks += wt * wt;
      walked += 1.f;
      m = mn;
      asm volatile("s_nop 3" : "+v"(pb[0])::"memory");   // (written by the vector ALU just now)
#pragma unroll
      for (int k = 0; k < 2 * NV; ++k) {
        if (k == NV) asm volatile("s_nop 3" : "+v"(pb[1])::"memory");
        mma_acc(o[k % NV], vf[k % AHEAD], pb[k / NV]);
        if (k + AHEAD < 2 * NV) vf[k % AHEAD] = vfrag(cur * IMG, (k + AHEAD) % NV, (k + AHEAD) / NV);
        if (k < NV) weights(8 + k / 4 * 2, k % 4);   // the second half's, beside the first half's products
        if (MW == 0 && k >= 14 && k % 2 == 0) dma((k - 14) / 2);
        __builtin_amdgcn_sched_barrier(0);
      }
      {
        auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(ps), __float_as_uint(ps), false, false);
        lsum += __uint_as_float(w[0]) + __uint_as_float(w[1]);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (two[j]) {   // what rounding took from the weights of these 16 keys
#pragma unroll
          for (int v = 0; v < AHEAD; ++v) vf[v] = vfrag(cur * IMG, v, j);
          bf16x8 pr;
          float rs = 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            pr[i] = (bf16)(p[8 * j + i] - (float)pb[j][i]);
            rs += (float)pr[i];
          }
          auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(rs), __float_as_uint(rs), false, false);
          lsum += __uint_as_float(w[0]) + __uint_as_float(w[1]);
          asm volatile("s_nop 3" : "+v"(pr)::"memory");
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            mma_acc(o[v], vf[v % AHEAD], pr);
            if (v + AHEAD < NV) vf[v % AHEAD] = vfrag(cur * IMG, v + AHEAD, j);
          }
        }
      cur = nxt;
      if (MW == 0) landed(true);   // (tile n + 2)
      __syncthreads();
    }
    asm volatile(MMA_WAIT "\n\ts_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // ---- epilogue: O^T lane map dim = 32 v + 8 (i / 4) + 4 hf + i % 4, row = col ----
    const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
    if (my_parts == 1 && NW == 4 && !DECODE) {
      // through LDS (the images are done with): 32 rows x 256 dims at a time, so that rows leave in 512-byte runs
      // instead of 8-byte pieces (prompts of 128-row tiles 3..5% faster; lower tiles and decode steps not)
      constexpr int LD = DV / 2 + 8;   // padded row
      static_assert(NW * 32 * LD * 2 <= (int)sizeof(sK), "the output fits the images");
      bf16* so = reinterpret_cast<bf16*>(sK) + wave * 32 * LD;
      const uint64_t own = __ballot(mine);
      const int64_t place = (int64_t)t * out_stride_t + (int64_t)head * DV;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the first half's reads
#pragma unroll
        for (int v = 0; v < NV / 2; ++v)
#pragma unroll
          for (int i = 0; i < 16; i += 4) {
            const f32x16& x = o[half * (NV / 2) + v];
            *reinterpret_cast<bf16x4*>(so + col * LD + 32 * v + 2 * i + 4 * hf) =
                bf16x4{(bf16)(x[i] * inv), (bf16)(x[i + 1] * inv), (bf16)(x[i + 2] * inv), (bf16)(x[i + 3] * inv)};
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (a wave's own rows: no barrier)
#pragma unroll 4
        for (int i = 0; i < 16; ++i) {
          // the row's place from the lane that holds it: divided out again for each row, the output took 5.1 us of a tile's life instead of 3.7
          const int lr = 2 * i + hf;
          const uint32_t lo = __builtin_amdgcn_ds_bpermute(4 * lr, (int)(uint32_t)place), hi = __builtin_amdgcn_ds_bpermute(4 * lr, (int)(uint32_t)(place >> 32));
          const bf16x8 x = ld8(so + lr * LD + 8 * col);
          if ((own >> lr) & 1) st8(out + (int64_t)((uint64_t)hi << 32 | lo) + half * (DV / 2) + 8 * col, x);
        }
      }
    } else if (!mine) {
      // written by its own pass
    } else if (my_parts == 1) {
      bf16* op = out + (int64_t)t * out_stride_t + (int64_t)head * DV + 4 * hf;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < 16; i += 4)
          *reinterpret_cast<bf16x4*>(op + 32 * v + 2 * i) = bf16x4{(bf16)(o[v][i] * inv), (bf16)(o[v][i + 1] * inv),
                                                                   (bf16)(o[v][i + 2] * inv), (bf16)(o[v][i + 3] * inv)};
    } else {   // partials in the lanes' own order: 1 KiB a store (mla_reduce_rows_kernel reads them so)
      const int64_t slot = DECODE ? blockIdx.x : (int64_t)unit * parts + part;
      float* wp = ws_o + (slot * NW + wave) * (32 * DV) + 4 * lane;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < 16; i += 4)
          *reinterpret_cast<f32x4*>(wp + (4 * v + i / 4) * 256) =
              f32x4{o[v][i] * inv, o[v][i + 1] * inv, o[v][i + 2] * inv, o[v][i + 3] * inv};
      if (hf == 0) {
        ws_ml[2 * (slot * RT + wave * 32 + col)] = m;
        ws_ml[2 * (slot * RT + wave * 32 + col) + 1] = lsum;
      }
    }
  };
  const int bt0 = __builtin_amdgcn_readlane(tl_row, __builtin_ctzll(left));
  const bool same0 = ((left >> lane) & 1) && tl_row == bt0;
  left &= ~__ballot(same0);
  walk(bt0, same0, lane);
  if (MW > 0 && wave >= NW) return;
  // Tokens of further block-table rows: an `own_seq` workgroup takes them, unless they are not in order.  (Those go one
  // row at a time: a second pass here would hold its operands over the first one's epilogue, in scratch.)
  if constexpr (!DECODE) {
    for (; left; left &= left - 1) {
      const int at = __builtin_ctzll(left), bt_row = __builtin_amdgcn_readlane(tl_row, at), tok = t0 + at;
      const int first = t0 + __builtin_ctzll(__ballot(lane < nt && tl_row == bt_row));
      if (bt_row > 0 && bt_row < seqs && first_token(tok_row, T, bt_row) == first) continue;
      const int lo = max(row0 + wave * 32, tok * H), hi = min(min(row0 + wave * 32 + 32, row_end), (tok + 1) * H);
      for (int row = lo; row < hi; ++row)
        plain_row<DK, DV>(q + (int64_t)tok * q_stride_t + (int64_t)(row - tok * H) * DK, cache, block_tables + (int64_t)bt_row * bt_stride,
                          part == 0 ? kv_lens[tok] : 0, scale_log2, my_parts == 1,
                          out + (int64_t)tok * out_stride_t + (int64_t)(row - tok * H) * DV,
                          ws_o + (((int64_t)unit * parts + part) * NW + wave) * (32 * DV) + 4 * ((row - row0) & 31),
                          ws_ml + 2 * (((int64_t)unit * parts + part) * RT + row - row0));
    }
  }
}

// Merge the partials of row tiles: a wave of (tile, 32 rows, 32 value dims) per quarter, lanes as the tile kernel's, 1 KiB a
// load; partials eight at a time with their loads issued up front, as below.
template <int DV, int NW>
__global__ __launch_bounds__(256) void mla_reduce_rows_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                              int T, int H, int parts, const int2* __restrict__ plan,
                                                              bf16* __restrict__ out, int64_t out_stride_t) {
  constexpr int RT = 32 * NW;
  const int unit = blockIdx.x / NW, wave = blockIdx.x % NW, v = blockIdx.y, qd = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int col = lane & 31, hf = lane >> 5, HG = (H + RT - 1) / RT;
  int64_t base = (int64_t)unit * parts;
  if (plan != nullptr) {
    const int2 pl = plan[unit];
    base = pl.x;
    parts = pl.y;
    if (parts == 1) return;   // written by its one piece
  }
  const int row = (plan ? unit / HG * H + unit % HG * RT : unit * RT) + wave * 32 + col;
  if (row >= (plan ? (unit / HG + 1) * H : T * H)) return;
  float M = OME_NEG_INF, den = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < parts; p0 += 8) {
    float mm[8], ll[8];
    f32x4 vv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t r = base + min(p0 + j, parts - 1);
      mm[j] = ws_ml[2 * (r * RT + wave * 32 + col)];
      ll[j] = p0 + j < parts ? ws_ml[2 * (r * RT + wave * 32 + col) + 1] : 0.f;
      vv[j] = *reinterpret_cast<const f32x4*>(ws_o + (r * NW + wave) * (32 * DV) + (4 * v + qd) * 256 + 4 * lane);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (!(ll[j] > 0.f)) continue;
      const float mn = fmaxf(M, mm[j]);
      const float a = __builtin_amdgcn_exp2f(M - mn), w = ll[j] * __builtin_amdgcn_exp2f(mm[j] - mn);
      acc = acc * a + w * vv[j];
      den = den * a + w;
      M = mn;
    }
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  const int t = row / H;
  *reinterpret_cast<bf16x4*>(out + (int64_t)t * out_stride_t + (int64_t)(row - t * H) * DV + 32 * v + 8 * qd + 4 * hf) =
      bf16x4{(bf16)(acc[0] * inv), (bf16)(acc[1] * inv), (bf16)(acc[2] * inv), (bf16)(acc[3] * inv)};
}

// ------------------------------------------------------------------------------------------
// Many decode rows of 128 heads: one workgroup of 8 waves owns a token's heads and one partition of its keys.  A wave owns
// 16 heads and all DV value dims, so two waves share a SIMD: less matrix work an LDS read than the row tiles above,
// but a piece's start, drain and tile reads overlap with another wave's work, which counts where contexts are short and
// pieces many.  Row tiles -> these: 64 / 128 / 256 rows of ~400 keys 50 -> 44, 64 -> 56, 73 -> 69 us; 48 rows of ~3000
// 86 -> 94.
// Key tiles arrive by LDS DMA into a double-buffered image: the DMA of tile n + 1 is issued before tile n is
// computed and retired (vmcnt(0) + barrier) after it.
// ------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void mla_lds_t;

template <int DK, int DV, int NW>
__global__ __launch_bounds__(64 * NW, 1) void mla_attn_all_kernel(
    const bf16* __restrict__ q, int64_t q_stride_t, const bf16* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_row,
    const int* __restrict__ kv_lens, int H, float scale_log2, int parts, bf16* __restrict__ out,
    int64_t out_stride_t, float* __restrict__ ws_o, float* __restrict__ ws_ml) {
  static_assert(DK == 576 && lds_chunks<DK>() == DK / 8, "LDS DMA image assumes unpadded 72-chunk rows");
  constexpr int CH = DK / 8, NI = KT * CH / 64, NB = DV / 16;
  constexpr int IMG = KT * CH * 8;   // bf16 elements per K-tile image
  __shared__ __attribute__((aligned(16))) bf16 sK[2 * IMG];
  const int t = blockIdx.x, part = blockIdx.z;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, g = lane >> 4;
  const int head = blockIdx.y * 16 * NW + wave * 16 + col;   // this lane's head (S^T / O^T column)
  const int L = kv_lens[t];
  const int n_pages = (L + 15) >> 4;
  const int pairs = (n_pages + 1) >> 1;
  const int per_part = (pairs + parts - 1) / parts;
  const int pair_begin = part * per_part, pair_end = min(pairs, pair_begin + per_part);
  const int* bt = block_tables + (int64_t)tok_row[t] * bt_stride;

  // K tile pair -> LDS image: instruction i writes chunks [64 i, 64 i + 64) lane-linearly, each
  // lane fetching the source chunk the row's XOR swizzle puts there.  A page is 16 rows x 72 chunks
  // = 18 instructions, so each instruction reads one page: its descriptor is based at that page.
  auto dma_pair = [&](int pr, bf16* img) {
#pragma unroll
    for (int j = 0; j < (NI + NW - 1) / NW; ++j) {
      const int i = wave + NW * j;
      if (i >= NI) break;
      const int c = 64 * i + lane, row = c / CH, xl = c - row * CH;
      const int pg = 2 * pr + (i >= NI / 2);
      const int page = bt[pg < n_pages ? pg : 0];
      const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)(cache + (int64_t)page * 16 * DK), (short)0,
                                                        16 * DK * 2, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (mla_lds_t*)(img + 64 * 8 * i), 16,
                                               (uint32_t)(((row & 15) * CH + (xl ^ (row & 7))) * 16), 0, 0, 0);
    }
  };
  if (pair_begin < pair_end) dma_pair(pair_begin, sK);

  bf16x8 qf[DK / 32];
  const bf16* qp = q + (int64_t)t * q_stride_t + (int64_t)head * DK + 8 * g;
#pragma unroll
  for (int s = 0; s < DK / 32; ++s) qf[s] = ld8(qp + 32 * s);

  f32x4 o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = OME_NEG_INF, lsum = 0.f;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // The XOR swizzle makes every LDS offset lane-dependent; split it so the compiler sees a lane
  // base plus an immediate: (8k + c) ^ z = 8k + (c ^ z) for c, z < 8.  S^T reads chunk 4 s + g of
  // row col (2 bases by s parity); V^T reads chunk 2 nb + pcol/2 of row 4 g + qrow (4 bases by
  // nb mod 4).  Rows 16..31 sit 16 * CH chunks further on with the same (row & 7).
  const int qrow = (lane & 15) >> 2, pcol = lane & 3;
  int sofs[2], vofs[4];
#pragma unroll
  for (int e = 0; e < 2; ++e) sofs[e] = (col * CH + ((4 * e + g) ^ (col & 7))) * 16;
  const int rv = 4 * g + qrow;
#pragma unroll
  for (int e = 0; e < 4; ++e) vofs[e] = (rv * CH + ((2 * e + (pcol >> 1)) ^ (rv & 7))) * 16 + (pcol & 1) * 8;
  int buf = 0;
  for (int pr = pair_begin; pr < pair_end; ++pr) {
    const bf16* img = sK + buf * IMG;
    // the other image's last readers passed the barrier that ended the previous tile
    if (pr + 1 < pair_end) dma_pair(pr + 1, sK + (buf ^ 1) * IMG);
    // ---- S^T [32 keys x 16 heads] ----
    const char* ib = reinterpret_cast<const char*>(img);
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) {
      const int off = sofs[s & 1] + (s >> 1) * 128;   // swz(col, 4 s + g): lane base + immediate
      const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(ib + off);
      const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(ib + off + 16 * CH * 16);
      s0 = mfma16x32(a0, qf[s], s0);
      s1 = mfma16x32(a1, qf[s], s1);
    }
    const int kbase = pr * KT;
    float mx = OME_NEG_INF;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s0[i] = (kbase + 4 * g + i < L) ? s0[i] * scale_log2 : OME_NEG_INF;
      s1[i] = (kbase + 16 + 4 * g + i < L) ? s1[i] * scale_log2 : OME_NEG_INF;
      mx = fmaxf(mx, fmaxf(s0[i], s1[i]));
    }
    mx = group4_max(mx);
    const float m_new = fmaxf(m, mx);
    const float alpha = (m_new == OME_NEG_INF) ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
    bf16x8 pb;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p0 = (m_new == OME_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(s0[i] - m_new);
      const float p1 = (m_new == OME_NEG_INF) ? 0.f : __builtin_amdgcn_exp2f(s1[i] - m_new);
      ps += p0 + p1;
      pb[i] = (bf16)p0;
      pb[4 + i] = (bf16)p1;
    }
    ps = group4_sum(ps);
    lsum = lsum * alpha + ps;
    m = m_new;
    // ---- O^T [DV x 16 heads] += V^T . P^T (keys permuted as in pb: 4g + i, 16 + 4g + i) ----
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int off = vofs[nb & 3] + (nb >> 2) * 128;   // swz(4g + qrow, 2 nb + pcol/2) + 8 (pcol & 1)
      const bf16x4 va = tr_read(img, off);
      const bf16x4 vb = tr_read(img, off + 16 * CH * 16);
      bf16x8 a;
      a[0] = va[0]; a[1] = va[1]; a[2] = va[2]; a[3] = va[3];
      a[4] = vb[0]; a[5] = vb[1]; a[6] = vb[2]; a[7] = vb[3];
      o[nb] *= alpha;
      o[nb] = mfma16x32(a, pb, o[nb]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile's DMA has landed
    __syncthreads();
    buf ^= 1;
  }

  // ---- epilogue: O^T lane map dim = 16 nb + 4 g + i, head = col ----
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (parts == 1) {
    bf16* op = out + (int64_t)t * out_stride_t + (int64_t)head * DV + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(o[nb][i] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * nb) = v;
    }
  } else {
    const int64_t ws_row = ((int64_t)t * H + head) * parts + part;
    float* wp = ws_o + ws_row * DV + 4 * g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      *reinterpret_cast<f32x4*>(wp + 16 * nb) = f32x4{o[nb][0] * inv, o[nb][1] * inv, o[nb][2] * inv,
                                                       o[nb][3] * inv};
    if (g == 0) {
      ws_ml[2 * ws_row] = m;
      ws_ml[2 * ws_row + 1] = lsum;
    }
  }
}

// merge split-K partitions: one workgroup per (token, head), DV / 4 threads x 4 dims.  Partitions
// are consumed 8 at a time with all their loads issued up front (online max rescaling), so up to
// 64 partitions cost ~8 memory latencies rather than one each.  Of more than 16 the empty ones are not read (nor
// written; loading the first 16 ahead of the length was slower, 15.4 instead of 14.5 us at 1000 keys).
template <int DV>
__global__ __launch_bounds__(128) void mla_reduce_kernel(const float* __restrict__ ws_o,
                                                         const float* __restrict__ ws_ml, int H, int parts,
                                                         bf16* __restrict__ out, int64_t out_stride_t,
                                                         const float* __restrict__ sinks, const int* __restrict__ kv_lens,
                                                         int window, int least, const int2* __restrict__ plan) {
  const int t = blockIdx.x, h = blockIdx.y;
  int64_t row0 = ((int64_t)t * H + h) * parts;
  int step = 1;
  if (plan != nullptr) {   // a token's pieces by length, 16 rows each
    const int2 pl = plan[t];
    parts = pl.y;
    if (parts == 1) return;   // written by its one piece
    row0 = (int64_t)pl.x * 16 + h;
    step = 16;
  } else if (parts > 16 && least > 0) {   // as the 16-head kernels cut them, `least` tiles and more (with 16 the empty ones cost less than the length's way here)
    const int L = kv_lens[t], tiles = ((L + 15) / 16 + 1) / 2 - (window > 0 ? max(L - window, 0) / KT : 0);
    const int live = live_parts(tiles, parts), per = tiles > 0 ? max(least, (tiles + live - 1) / live) : 0;
    parts = per > 0 ? (tiles + per - 1) / per : 0;
  }
  float M = OME_NEG_INF, den = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < parts; p0 += 8) {
    float mm[8], ll[8];
    f32x4 vv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t r = row0 + (int64_t)min(p0 + j, parts - 1) * step;
      mm[j] = ws_ml[2 * r];
      ll[j] = p0 + j < parts ? ws_ml[2 * r + 1] : 0.f;
      vv[j] = *reinterpret_cast<const f32x4*>(ws_o + r * DV + 4 * threadIdx.x);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (!(ll[j] > 0.f)) continue;
      const float mn = fmaxf(M, mm[j]);
      const float a = __builtin_amdgcn_exp2f(M - mn), w = ll[j] * __builtin_amdgcn_exp2f(mm[j] - mn);
      acc = acc * a + w * vv[j];
      den = den * a + w;
      M = mn;
    }
  }
  if (sinks != nullptr) {
    const float sk = sinks[h] * 1.4426950408889634f;
    const float mn = fmaxf(M, sk), a = __builtin_amdgcn_exp2f(M - mn);
    acc = acc * a;
    den = den * a + __builtin_amdgcn_exp2f(sk - mn);
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  bf16x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (bf16)(acc[i] * inv);
  *reinterpret_cast<bf16x4*>(out + (int64_t)t * out_stride_t + (int64_t)h * DV + 4 * threadIdx.x) = r;
}

// q [T, H, DK] (token stride q_stride_t), cache [pages, 16, DK], out [T, H, DV] with
// (DK, DV) = (576, 512) or (288, 256).  tok_row[t] = block-table row of token t; kv_lens[t] =
// keys visible to token t (causal).  parts > 1 needs ws_o [R*DV] f32 and ws_ml [R*2] f32, R = T*H*parts; of row
// tiles (`rows`) whole tiles: R = ceil(T*H / rows)*rows*parts for prompts, and for decode (`plan`, int2 [256], written
// by the kernel) 256*rows, one tile a piece.
template <int DK, int DV>
static void mla_launch(const void* q, int64_t q_stride_t, const void* cache, const int* block_tables, int bt_stride,
                       const int* tok_row, const int* kv_lens, int T, int H, float scale_log2, int parts, void* out,
                       int64_t out_stride_t, float* ws_o, float* ws_ml, hipStream_t stream, int rows = 0, int seqs = 1,
                       int2* plan = nullptr, const float* sinks = nullptr, int window = -1) {
  // `rows`: query rows of a workgroup of the row-tile kernel (32 / 64 / 128, the caller's choice), 0: the
  // 16-head kernel, which alone has the sink term and the window, or many rows of 128 heads
  if (rows > 0 && !(scale_log2 > 0.f)) rows = 0, parts = 1;   // (row tiles look for the largest score before they scale it)
  if constexpr (DK == 576) {
    if (rows > 0) {
      const unsigned units = (unsigned)(plan ? T * ((H + rows - 1) / rows) : ((int64_t)T * H + rows - 1) / rows);
      const dim3 grid(plan && parts > 1 ? 256 : units + (plan || seqs < 2 ? 0 : seqs - 1), plan ? 1 : parts);
#define MLA_ROWS(NW)                                                                                                    \
  {                                                                                                                      \
    const auto kernel = plan ? mla_attn_rows_kernel<DK, DV, NW, true> : mla_attn_rows_kernel<DK, DV, NW, false>;          \
    kernel<<<grid, 64 * (NW + row_movers(NW)), 0, stream>>>((const bf16*)q, q_stride_t, (const bf16*)cache, block_tables, bt_stride,         \
                                         tok_row, kv_lens, T, H, seqs, scale_log2, parts, plan, (bf16*)out,               \
                                         out_stride_t, ws_o, ws_ml);                                                     \
    if (parts > 1)                                                                                                       \
      mla_reduce_rows_kernel<DV, NW><<<dim3(units * NW, DV / 32), 256, 0, stream>>>(ws_o, ws_ml, T, H, parts, plan,       \
                                                                                    (bf16*)out, out_stride_t);            \
  }
      if (rows == 32 && plan && H <= 16 && (int64_t)T * bt_stride >= 3000) {
        mla_attn_pages_kernel<DK, DV, true><<<parts > 1 ? 256 : T, 256, 0, stream>>>(
            (const bf16*)q, q_stride_t, (const bf16*)cache, block_tables, bt_stride, tok_row, kv_lens, T, H, scale_log2, parts, plan,
            (bf16*)out, out_stride_t, ws_o, ws_ml, nullptr, -1);
        if (parts > 1)
          mla_reduce_kernel<DV><<<dim3(T, H), DV / 4, 0, stream>>>(ws_o, ws_ml, H, parts, (bf16*)out, out_stride_t, nullptr, kv_lens, -1, 0, plan);
      }
      else if (rows == 128) MLA_ROWS(4)
      else if (rows == 64) MLA_ROWS(2)
      else MLA_ROWS(1)
#undef MLA_ROWS
      return;
    }
  }
  bool done = false;
  if constexpr (DK == 576) {
    if (H % 128 == 0 && T >= 64 && sinks == nullptr && window <= 0) {   // (MLAWorkspace.parts cuts for it)
      mla_attn_all_kernel<DK, DV, 8><<<dim3(T, H / 128, parts), 512, 0, stream>>>(
          (const bf16*)q, q_stride_t, (const bf16*)cache, block_tables, bt_stride, tok_row, kv_lens, H, scale_log2,
          parts, (bf16*)out, out_stride_t, ws_o, ws_ml);
      done = true;
    }
  }
  if constexpr (DK == 576) {
    // (few workgroups over short tables: the old kernel starts a microsecond sooner.  It also has a CU hold several workgroups)
    const int64_t wgs = (int64_t)T * ((H + 15) / 16);
    if (!done && wgs * parts <= 512 && (wgs > 16 || bt_stride > 96)) {
      mla_attn_pages_kernel<DK, DV, false><<<dim3(T, (H + 15) / 16, parts), 256, 0, stream>>>(
          (const bf16*)q, q_stride_t, (const bf16*)cache, block_tables, bt_stride, tok_row, kv_lens, T, H, scale_log2,
          parts, nullptr, (bf16*)out, out_stride_t, ws_o, ws_ml, sinks, window);
      if (parts > 1)
        mla_reduce_kernel<DV><<<dim3(T, H), DV / 4, 0, stream>>>(ws_o, ws_ml, H, parts, (bf16*)out, out_stride_t, sinks, kv_lens, window, LEAST_PAIRS, nullptr);
      return;
    }
  }
  if (!done)
    mla_attn_kernel<DK, DV><<<dim3(T, (H + 15) / 16, parts), 256, 0, stream>>>(
        (const bf16*)q, q_stride_t, (const bf16*)cache, block_tables, bt_stride, tok_row, kv_lens, H, scale_log2,
        parts, (bf16*)out, out_stride_t, ws_o, ws_ml, sinks, window);
  if (parts > 1)
    mla_reduce_kernel<DV><<<dim3(T, H), DV / 4, 0, stream>>>(ws_o, ws_ml, H, parts, (bf16*)out, out_stride_t, sinks, kv_lens, window, done ? 0 : 1, nullptr);
}

OME_API int ome_mla_attn(const void* q, int64_t q_stride_t, const void* cache, const int* block_tables,
                         int bt_stride, int seqs, const int* tok_row, const int* kv_lens, int T, int H, int dk, int dv,
                         float scale, int parts, int rows, void* plan, void* out, int64_t out_stride_t, float* ws_o,
                         float* ws_ml, hipStream_t stream) {
  if (T <= 0) return 0;
  if ((rows != 0 && rows != 32 && rows != 64 && rows != 128) || (int64_t)T * H > 0x7fffff00 || parts > 65535) return -2;
  if (rows != 0 && (dk != 576 || dv != 512 || H < 4 || (uintptr_t)out % 16 || out_stride_t % 8)) return -2;
  if (plan && (rows == 0 || (parts > 1 && (int64_t)T * ((H + rows - 1) / rows) > 256))) return -2;   // (256 pieces)
  if (H <= 0 || parts < 1 || (parts > 1 && (!ws_o || !ws_ml))) return -2;
  const float scale_log2 = scale * 1.4426950408889634f;
  if (dk == 576 && dv == 512)
    mla_launch<576, 512>(q, q_stride_t, cache, block_tables, bt_stride, tok_row, kv_lens, T, H, scale_log2, parts, out,
                         out_stride_t, ws_o, ws_ml, stream, rows, seqs, (int2*)plan);
  else if (dk == 288 && dv == 256)
    mla_launch<288, 256>(q, q_stride_t, cache, block_tables, bt_stride, tok_row, kv_lens, T, H, scale_log2, parts, out,
                         out_stride_t, ws_o, ws_ml, stream, rows, seqs, (int2*)plan);
  else
    return -3;
  OME_CHECK_LAUNCH();
  return 0;
}

// Latent attention over rows of any latent / rotary width, padded to the kernel's tiling: a cache
// row is [latent (dv_pad wide: the values, zero beyond the latent) | rotary key (dk - dv_pad wide,
// zero beyond it)], dv_pad a multiple of 64 up to 256 or 512, dk - dv_pad 32 or 64.  Kernels as for
// ome_mla_attn; sinks optional, window > 0: a token sees only the last `window` of its kv_lens keys (both by the
// 16-head kernel).  Zero columns add nothing to a score, and the output's zero columns are dropped by
// the caller.
OME_API int ome_latent_attn(const void* q, int64_t q_stride_t, const void* cache, const int* block_tables,
                            int bt_stride, int seqs, const int* tok_row, const int* kv_lens, int T, int H, int dk, int dv,
                            float scale, int parts, int rows, void* plan, void* out, int64_t out_stride_t, float* ws_o,
                            float* ws_ml, const float* sinks, int window, hipStream_t stream) {
  if (T <= 0) return 0;
  if ((rows != 0 && rows != 32 && rows != 64 && rows != 128) || (int64_t)T * H > 0x7fffff00 || parts > 65535) return -2;
  if (rows != 0 && (sinks || window > 0)) return -2;
  if (rows != 0 && (dk != 576 || dv != 512 || H < 4 || (uintptr_t)out % 16 || out_stride_t % 8)) return -2;
  if (plan && (rows == 0 || (parts > 1 && (int64_t)T * ((H + rows - 1) / rows) > 256))) return -2;   // (256 pieces)
  if (H <= 0 || parts < 1 || (parts > 1 && (!ws_o || !ws_ml))) return -2;
  const float scale_log2 = scale * 1.4426950408889634f;
#define LATENT_CASE(DK_, DV_)                                                                                       \
  if (dk == DK_ && dv == DV_) {                                                                                     \
    mla_launch<DK_, DV_>(q, q_stride_t, cache, block_tables, bt_stride, tok_row, kv_lens, T, H, scale_log2, parts,  \
                         out, out_stride_t, ws_o, ws_ml, stream, rows, seqs, (int2*)plan, sinks, window);                                \
    OME_CHECK_LAUNCH();                                                                                             \
    return 0;                                                                                                       \
  }
  LATENT_CASE(96, 64)
  LATENT_CASE(128, 64)
  LATENT_CASE(160, 128)
  LATENT_CASE(192, 128)
  LATENT_CASE(224, 192)
  LATENT_CASE(256, 192)
  LATENT_CASE(288, 256)
  LATENT_CASE(320, 256)
  LATENT_CASE(544, 512)
  LATENT_CASE(576, 512)
#undef LATENT_CASE
  return -3;
}

// ------------------------------------------------------------------------------------------
// MLA pre-attention glue as ONE launch per layer (it was ~25 PyTorch elementwise / cat /
// index_select / index_copy kernels per layer: profiles/r03_deepseek_v3_fp8_reduced.md "other").
// One workgroup per token t:
//   cache[slot_t][0 : lat]          = RMSNorm(a[t, qlr : qlr + lat]) * w       (kv_a_layernorm)
//   cache[slot_t][lat : lat + rope] = RoPE_pos(a[t, qlr + lat : qlr + lat + rope])
//   qf[t, h, lat : lat + rope]      = RoPE_pos(q[t, h, nope : nope + rope])   for every head h
// RoPE in NeoX halves (the checkpoint's interleaved rows are permuted at load), table cs[pos] =
// [cos | sin] fp32; fp32 math, bf16 stores (the reference op's order: x * rs * w, rounded once).
// Padding rows (slot < 0) write row 0 of the scratch page, as the eager path did.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void mla_prep_kernel(const bf16* __restrict__ a, int64_t lda, int qlr, int lat,
                                                       int rope, const bf16* __restrict__ w, float eps,
                                                       const int* __restrict__ pos, const float* __restrict__ cs,
                                                       const int* __restrict__ slots, bf16* __restrict__ cache,
                                                       int64_t cache_row, const bf16* __restrict__ q, int64_t q_tok,
                                                       int64_t q_head, int nope, int H, bf16* __restrict__ qf,
                                                       int64_t qf_tok, int64_t qf_head) {
  __shared__ float red[4];
  const int t = blockIdx.x, tid = threadIdx.x;
  const bf16* ar = a + (int64_t)t * lda + qlr;
  int slot = slots[t];
  slot = slot < 0 ? 0 : slot;
  bf16* crow = cache + (int64_t)slot * cache_row;
  float ss = 0.f;
  for (int i = tid; i < lat; i += 256) {
    const float v = (float)ar[i];
    ss += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float rs = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)lat + eps);
  for (int i = tid; i < lat; i += 256) crow[i] = (bf16)((float)ar[i] * rs * (float)w[i]);
  const int half = rope >> 1;
  const float* c = cs + (int64_t)pos[t] * rope;
  // k_pe: pairs (j, j + half)
  for (int j = tid; j < half; j += 256) {
    const float x1 = (float)ar[lat + j], x2 = (float)ar[lat + half + j];
    const float co = c[j], si = c[half + j];
    crow[lat + j] = (bf16)(x1 * co - x2 * si);
    crow[lat + half + j] = (bf16)(x2 * co + x1 * si);
  }
  // q_pe of every head
  for (int k = tid; k < H * half; k += 256) {
    const int h = k / half, j = k - h * half;
    const bf16* qr = q + (int64_t)t * q_tok + (int64_t)h * q_head + nope;
    const float x1 = (float)qr[j], x2 = (float)qr[half + j];
    const float co = c[j], si = c[half + j];
    bf16* o = qf + (int64_t)t * qf_tok + (int64_t)h * qf_head + lat;
    o[j] = (bf16)(x1 * co - x2 * si);
    o[half + j] = (bf16)(x2 * co + x1 * si);
  }
}

OME_API int ome_mla_prep(const void* a, int64_t lda, int qlr, int lat, int rope, const void* w, float eps,
                         const int* pos, const float* cs, const int* slots, void* cache, int64_t cache_row,
                         const void* q, int64_t q_tok, int64_t q_head, int nope, int H, void* qf, int64_t qf_tok,
                         int64_t qf_head, int T, hipStream_t stream) {
  if (T <= 0) return 0;
  if (rope % 2 || lat <= 0 || H <= 0) return -2;
  mla_prep_kernel<<<T, 256, 0, stream>>>((const bf16*)a, lda, qlr, lat, rope, (const bf16*)w, eps, pos, cs, slots,
                                         (bf16*)cache, cache_row, (const bf16*)q, q_tok, q_head, nope, H, (bf16*)qf,
                                         qf_tok, qf_head);
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Latent-attention glue (any latent width / rotary width, bf16 or fp32): the absorbed form is
// multi-query attention with ONE shared head whose key is [RMSNorm(c) * w | rotated k_pe] and whose
// value is the latent RMSNorm(c) * w itself.  From the fused down-projection output a [T, qlr + lat
// + rope] this writes, per token, the key row  k_cache[slot, 0 : lat] = latent,  k_cache[slot,
// rope_off : rope_off + rope] = rotated k_pe  (rows D wide, rope_off >= lat; the gaps are never
// written: the caches start as zeros) and -- only for the generic paged attention kernels, which
// read values from their own array -- the value column v_cache[page, 0, 0 : lat, off]; the latent
// kernel (ome_latent_attn) takes its values from the key rows, so v_cache is nullptr there.  For
// every head the rotated q_pe goes to qf[t, h, rope_off : rope_off + rope], zeros into the gaps up
// to D.  Rotary pairs are (j, j + rope/2), angles from the fp32 table row of the token's position
// (cos | sin, any frequency scaling baked in).  k_cache == nullptr: a layer that reads another
// layer's cache only rotates its queries.  Padding rows (slot < 0) write slot 0 of the scratch page.
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void latent_prep_kernel(
    const T* __restrict__ a, int64_t lda, int qlr, int lat, int rope, const T* __restrict__ w, float eps,
    const int* __restrict__ pos, const float* __restrict__ cs, const int* __restrict__ slots,
    T* __restrict__ k_cache, T* __restrict__ v_cache, int D, int P, int rope_off, const T* __restrict__ q,
    int64_t q_tok, int64_t q_head, int nope, int H, T* __restrict__ qf, int64_t qf_tok, int64_t qf_head) {
  __shared__ float red[4];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int half = rope >> 1;
  const float* c = cs + (int64_t)pos[t] * rope;
  if (k_cache != nullptr) {
    const T* ar = a + (int64_t)t * lda + qlr;
    int slot = slots[t];
    slot = slot < 0 ? 0 : slot;
    T* krow = k_cache + (int64_t)slot * D;
    T* vcol = v_cache != nullptr ? v_cache + (int64_t)(slot / P) * D * P + slot % P : nullptr;
    float ss = 0.f;
    for (int i = tid; i < lat; i += 256) {
      const float v = (float)ar[i];
      ss += v * v;
    }
    ss = block_sum<256>(ss, red);
    const float rs = 1.f / sqrtf(ss / (float)lat + eps);
    for (int i = tid; i < lat; i += 256) {
      const T v = (T)((float)ar[i] * rs * (float)w[i]);
      krow[i] = v;
      if (vcol != nullptr) vcol[(int64_t)i * P] = v;
    }
    for (int j = tid; j < half; j += 256) {
      const float x1 = (float)ar[lat + j], x2 = (float)ar[lat + half + j];
      const float co = c[j], si = c[half + j];
      krow[rope_off + j] = (T)(x1 * co - x2 * si);
      krow[rope_off + half + j] = (T)(x2 * co + x1 * si);
    }
  }
  const int gap = rope_off - lat, tail = D - rope_off - rope;
  for (int k = tid; k < H * half; k += 256) {
    const int h = k / half, j = k - h * half;
    const T* qr = q + (int64_t)t * q_tok + (int64_t)h * q_head + nope;
    const float x1 = (float)qr[j], x2 = (float)qr[half + j];
    const float co = c[j], si = c[half + j];
    T* o = qf + (int64_t)t * qf_tok + (int64_t)h * qf_head + rope_off;
    o[j] = (T)(x1 * co - x2 * si);
    o[half + j] = (T)(x2 * co + x1 * si);
  }
  for (int k = tid; k < H * (gap + tail); k += 256) {
    const int h = k / (gap + tail), j = k - h * (gap + tail);
    qf[(int64_t)t * qf_tok + (int64_t)h * qf_head + (j < gap ? lat + j : rope_off + rope + j - gap)] = (T)0.f;
  }
}

OME_API int ome_latent_prep(const void* a, int64_t lda, int qlr, int lat, int rope, const void* w, float eps,
                            const int* pos, const float* cs, const int* slots, void* k_cache, void* v_cache, int D,
                            int P, int rope_off, const void* q, int64_t q_tok, int64_t q_head, int nope, int H,
                            void* qf, int64_t qf_tok, int64_t qf_head, int T, int f32, hipStream_t stream) {
  if (T <= 0) return 0;
  if (rope % 2 || lat <= 0 || H <= 0 || rope_off < lat || rope_off + rope > D || P <= 0) return -2;
  if (f32)
    latent_prep_kernel<float><<<T, 256, 0, stream>>>((const float*)a, lda, qlr, lat, rope, (const float*)w, eps, pos,
                                                     cs, slots, (float*)k_cache, (float*)v_cache, D, P, rope_off,
                                                     (const float*)q, q_tok, q_head, nope, H, (float*)qf, qf_tok,
                                                     qf_head);
  else
    latent_prep_kernel<bf16><<<T, 256, 0, stream>>>((const bf16*)a, lda, qlr, lat, rope, (const bf16*)w, eps, pos, cs,
                                                    slots, (bf16*)k_cache, (bf16*)v_cache, D, P, rope_off,
                                                    (const bf16*)q, q_tok, q_head, nope, H, (bf16*)qf, qf_tok,
                                                    qf_head);
  return (int)hipGetLastError();
}
