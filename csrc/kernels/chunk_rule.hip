// Prompt rows of the matrix-state layers with one decay per head, in chunks of 32 rows on the matrix
// cores (gfx950): the gated delta rule of Qwen3-Next / Jet-Nemotron (DELTA) and the selective scan of
// Mamba-2 (not DELTA).  With S [dk, dv] the state a chunk starts from, k_i / q_i its key and query
// rows (unit-norm for DELTA, B / C for Mamba-2), g_i = exp(cum_i) the decay from the chunk's start up to and
// with row i:
//   DELTA   A_ij = beta_i exp(cum_i - cum_j) k_i.k_j (j < i),  T = (I + A)^-1,
//           U = T R,  R_i = beta_i (v_i - g_i k_i S)                    Mamba-2   U_i = dt_i x_i
//   o_i = g_i q_i S + sum_{j <= i} P_ij U_j,  P_ij = exp(cum_i - cum_j) q_i.k_j     (+ D x_i)
//       (DELTA: P U = (P T) R, so that o and U both follow from R)
//   S'  = g_C S + sum_i exp(cum_C - cum_i) k_i U_i^T
//
// Two launches.  chunk_gram_kernel (Mamba-2: ssm_gram_kernel), parallel over all rows: the 32 x 32 matrices
// P T and T (Mamba-2: q k^T, which the heads of a group share) and the chunk's scalars, into a workspace.
// chunk_rule_kernel walks the chunks of a (sequence, head) in order: a wave owns 16 value columns and keeps its
// S in VGPR accumulators.
//
// What bounds it: the chain of chunks.  Two waves a SIMD (S, one chunk's rows in flight and the split
// parts fill the registers) share its matrix and vector units at about 60 matrix (DELTA: 96) and 500 vector
// instructions a chunk, near 3 us with the latencies between them; its memory traffic hides behind that (leaving
// the reads out gives 1%).  Per-head P, formed in the first launch, cost 40 us there and 108 in the scan
// (Mamba-2, below): written and read back it is 16 times the bytes of its group's q k^T.
//   gated delta rule, 32 heads of 128 x 128, prompts of 1001 / 1435 / 1564 rows:   24 + 123 us (row by row: 1098)
//   selective scan, 128 heads of 64 x 128, 8 groups, 1033 / 926 / 1248 / 293 rows:  11 + 116 us (row by row: 1745)
// Largest error of the state against 64 bits: 1.1e-7 (row by row: 2.0e-7) and 1.4e-7 (6.2e-7) of its norm.
//
// A chunk's products multiply the entries that causality zeroes as well, and 0 times an infinity or NaN is NaN, so a key,
// gate or value that is not finite would reach the rows before it in its chunk.  It reaches S and stays there (each
// U_i enters every channel of S, and no decay takes an infinity or NaN away), so S tells at the end of a sequence: a
// wave whose S is not finite walks its columns again row by row.
//
// fp32 throughout: k and q enter the matrix cores as the bf16 values that they are (their norms, 1 / |k| and
// 1 / (|q| sqrt(dk)), scale results), S and U as three bf16 parts that sum to the fp32 value exactly, at
// 3/16 of the fp32 MFMA's time; T R and P U, where both operands are fp32, take the fp32 MFMA.  Decay
// exponents are summed in fp64 (differences of a long sum).  The row-by-row kernels stay for decode steps
// (one row per sequence), few rows in all, dk other than 64 / 128, and unaligned views.
#include "common.h"

namespace {

constexpr int RC = 32;            // rows of a chunk
constexpr int LDM = RC + 4;       // padded row of a 32 x 32 fp32 matrix in LDS
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// workspace of one chunk.  DELTA, per head: P T, T, then the vectors a, b, c, d [32] and g_C.  Mamba-2, per group: q k^T
// (its heads differ in their decays only, which the scan applies: P itself would be 16 times the bytes); then
// per head the vectors a, cum's upper and lower parts, c, d and g_C.
constexpr int NV_DELTA = 4 * RC + 4, NV_SSM = 5 * RC + 4;
template <bool DELTA>
constexpr int vec_floats() { return DELTA ? NV_DELTA : NV_SSM; }
template <bool DELTA>
__host__ __device__ constexpr int64_t ws_floats(int H, int G) {
  return DELTA ? (int64_t)H * (2 * RC * RC + NV_DELTA) : (int64_t)G * RC * RC + (int64_t)H * NV_SSM;
}

struct RuleArgs {
  const bf16 *q, *k, *v;          // rows of stride `stride` (v: v_stride)
  int64_t stride, v_stride;
  const bf16 *a, *b;              // per-head rows: a | b (DELTA), dt (Mamba-2)
  int64_t ab_stride;
  const float *A, *D, *dt_bias;   // A_log (DELTA) / A, D (Mamba-2)
  float dt_min;
  float* ws;
  float* state;                   // [slots, H, dv, dk]
  bf16* out;
  int64_t out_stride;
  const int *cu, *slot, *reset;
  int S, H, Hk, dv;
};

// Sequences of at most FEW rows (the decode rows beside a prompt) are walked row by row instead: no chunk in the workspace,
// no products 1/32 full.  The walk is bound by its vector instructions, near 1 us a row and four waves a CU.  Chunks -> walk, in us,
// delta rule of 32 heads of 128 x 128 (selective scan of 128 of 64 x 128): 200 sequences of 1 row with a prompt of 40
// 224 -> 193 (365 -> 327), of 2000 259 -> 224 (416 -> 346); 64 of 2 rows 81 -> 70 (131 -> 118), of 3 81 -> 81
// (126 -> 130), of 4 81 -> 93 (127 -> 144); one of 3 rows 16 -> 11 (12 -> 10).
constexpr int FEW = 3;

// Chunk `id` of the launch -> (sequence, first row).  Sequence s owns ids cu[s] / 32 + s and up, one per
// chunk: ceil(len / 32) <= (cu[s + 1] / 32 + s + 1) - (cu[s] / 32 + s), so ids never overlap and stay
// below T / 32 + S.  Whole wave; false: an id that no chunk has, or of a sequence that is walked.
__device__ __forceinline__ bool chunk_of(int id, const int* cu, int S, int& r0, int& n) {
  const int lane = threadIdx.x & 63;
  int s = -1;
  for (int b = 0; b < S; b += 64) {
    const int i = b + lane;
    const int c = __popcll(__ballot(i < S && cu[min(i, S)] / RC + i <= id));
    s += c;
    if (c < 64) break;
  }
  if (s < 0) return false;
  r0 = cu[s] + (id - cu[s] / RC - s) * RC;
  n = min(RC, cu[s + 1] - r0);
  return n > 0 && cu[s + 1] - cu[s] > FEW;
}

__device__ __forceinline__ f32x4 mma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// eight fp32 values -> three bf16 vectors that sum to them exactly (8 bits of the mantissa each)
__device__ __forceinline__ void split3(f32x4 x0, f32x4 x1, bf16x8 (&p)[3]) {
  float r[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = x0[j], r[4 + j] = x1[j];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    u32x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t lo = __float_as_uint(r[2 * j]), hi = __float_as_uint(r[2 * j + 1]);
      w[j] = __builtin_amdgcn_perm(hi, lo, 0x07060302);   // the two upper halves
      if (t < 2) {
        r[2 * j] -= __uint_as_float(lo & 0xffff0000u);
        r[2 * j + 1] -= __uint_as_float(hi & 0xffff0000u);
      }
    }
    p[t] = __builtin_bit_cast(bf16x8, w);
  }
}

// LDS written by lanes of a wave, read by others of the same wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float softplus_rule(float x) { return x > 20.f ? x : log1pf(__expf(x)); }

// ---------------------------------------------------------------------------------------------
// One wave per (chunk, head).  The 16-byte row pieces that a lane loads are both operands of q k^T and
// k k^T (rows and columns of a 16 x 16 x 32 product have the same lane layout).  T by forward substitution: lane j
// keeps column j in registers and reads the rows of A from LDS as broadcasts.
// ---------------------------------------------------------------------------------------------
template <int DK>
__global__ __launch_bounds__(256) void chunk_gram_kernel(RuleArgs a) {
  constexpr int NS = DK / 32;
  __shared__ __attribute__((aligned(16))) float sA[4][RC * LDM];
  __shared__ double s_cum[4][RC];
  __shared__ float s_vec[4][3][RC];   // 1 / |k|, 1 / (|q| sqrt(dk)), beta
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int h = blockIdx.y * 4 + w;
  int r0, n;
  if (h >= a.H || !chunk_of(blockIdx.x, a.cu, a.S, r0, n)) return;   // whole wave; no block barrier below
  const int hk = h / (a.H / a.Hk);
  float* ws = a.ws + ((int64_t)blockIdx.x * a.H + h) * (2 * RC * RC + NV_DELTA);

  bf16x8 kf[2][NS], qf[2][NS];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const int64_t r = r0 + min(16 * rb + col, n - 1);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      kf[rb][s] = ld8(a.k + r * a.stride + hk * DK + 32 * s + 8 * g);
      qf[rb][s] = ld8(a.q + r * a.stride + hk * DK + 32 * s + 8 * g);
    }
  }
  // per-row scalars: lane i (and i + 32) holds row i
  const int row = lane & 31, rv = r0 + min(row, n - 1);
  const bool ok = row < n;
  const float ga = -__expf(a.A[h]) * softplus_rule((float)a.a[(int64_t)rv * a.ab_stride + h] + a.dt_bias[h]);   // log decay
  const float beta = 1.f / (1.f + __expf(-(float)a.b[(int64_t)rv * a.ab_stride + h]));
  double cum = ok ? (double)ga : 0.0;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const double up = __shfl_up(cum, o, 32);
    if (row >= o) cum += up;
  }
  const double total = __shfl(cum, 31);   // rows past the chunk's end add nothing
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sk += (float)kf[rb][s][j] * (float)kf[rb][s][j];
        sq += (float)qf[rb][s][j] * (float)qf[rb][s][j];
      }
    sk = group4_sum(sk);
    sq = group4_sum(sq);
    if (g == 0) {
      s_vec[w][0][16 * rb + col] = rsqrtf(sk + 1e-6f);
      s_vec[w][1][16 * rb + col] = rsqrtf(sq + 1e-6f) * rsqrtf((float)DK);
    }
  }
  if (lane < RC) {
    s_cum[w][row] = cum;
    s_vec[w][2][row] = beta;
  }
  wave_sync();
  const float ik = s_vec[w][0][row], iq = s_vec[w][1][row];
  if (lane < RC) {   // the chunk's vectors (zero past its end: such rows add nothing anywhere)
    float* vec = ws + 2 * RC * RC;
    const float gi = __expf((float)cum), up = __expf((float)(total - cum));
    vec[row] = ok ? beta : 0.f;
    vec[RC + row] = ok ? beta * gi * ik : 0.f;
    vec[2 * RC + row] = ok ? gi * iq : 0.f;
    vec[3 * RC + row] = ok ? up * ik : 0.f;
    if (row == 0) vec[4 * RC] = __expf((float)total);
  }
  f32x4 pm[2][2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      f32x4 qk = {0.f, 0.f, 0.f, 0.f}, kk = {0.f, 0.f, 0.f, 0.f};
      if (cb <= rb) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          qk = mma_bf16(qf[rb][s], kf[cb][s], qk);
          kk = mma_bf16(kf[rb][s], kf[cb][s], kk);
        }
      }
      const int j = 16 * cb + col;
      const double cj = s_cum[w][j];
      const float ikj = s_vec[w][0][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * rb + 4 * g + e;
        float p = 0.f, m = 0.f;
        if (j <= i && i < n) {
          const float dec = __expf((float)(s_cum[w][i] - cj)) * ikj;
          p = qk[e] * dec * s_vec[w][1][i];
          m = j < i ? kk[e] * dec * s_vec[w][0][i] * s_vec[w][2][i] : 0.f;
        }
        pm[rb][cb][e] = p;
        sA[w][i * LDM + j] = m;
      }
    }
  wave_sync();
  float t[RC];
#pragma unroll
  for (int i = 0; i < RC; ++i) {
    float acc[4] = {i == row ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < i; m += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&sA[w][i * LDM + m]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (m + e < i) acc[e] -= x[e] * t[m + e];
    }
    t[i] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
  if (lane < RC) {
#pragma unroll
    for (int i = 0; i < RC; ++i) ws[RC * RC + i * RC + row] = t[i];
  }
  // P T: T's columns go through LDS into the product's operand layout (k-slot of step e: row 4 g + e)
  wave_sync();
  if (lane < RC) {
#pragma unroll
    for (int i = 0; i < RC; ++i) sA[w][i * LDM + row] = t[i];
  }
  wave_sync();
  f32x4 tb[2][2];   // [row block][column block]
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int cb = 0; cb <= kb; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) tb[kb][cb][e] = sA[w][(16 * kb + 4 * g + e) * LDM + 16 * cb + col];
  wave_sync();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb <= rb; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) sA[w][(16 * rb + 4 * g + e) * LDM + 16 * cb + col] = pm[rb][cb][e];
  wave_sync();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = cb; kb <= rb; ++kb) {
        const f32x4 m = *reinterpret_cast<const f32x4*>(&sA[w][(16 * rb + col) * LDM + 16 * kb + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) d = mma_f32(m[e], tb[kb][cb][e], d);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ws[(16 * rb + 4 * g + e) * RC + 16 * cb + col] = d[e];
    }
}

// Mamba-2: one block per (chunk, group).  Wave 0 multiplies q k^T (lower triangle), every half wave takes heads.
template <int DK>
__global__ __launch_bounds__(256) void ssm_gram_kernel(RuleArgs a) {
  constexpr int NS = DK / 32;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, hk = blockIdx.y;
  int r0, n;
  if (!chunk_of(blockIdx.x, a.cu, a.S, r0, n)) return;   // the same in every wave
  float* ws = a.ws + blockIdx.x * ws_floats<false>(a.H, a.Hk);
  if (w == 0) {
    bf16x8 kf[2][NS], qf[2][NS];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t r = r0 + min(16 * rb + col, n - 1);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        kf[rb][s] = ld8(a.k + r * a.stride + hk * DK + 32 * s + 8 * g);
        qf[rb][s] = ld8(a.q + r * a.stride + hk * DK + 32 * s + 8 * g);
      }
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb <= rb; ++cb) {
        f32x4 qk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s) qk = mma_bf16(qf[rb][s], kf[cb][s], qk);
#pragma unroll
        for (int e = 0; e < 4; ++e) ws[hk * RC * RC + (16 * rb + 4 * g + e) * RC + 16 * cb + col] = qk[e];
      }
  }
  const int row = lane & 31, rv = r0 + min(row, n - 1), per = a.H / a.Hk;
  const bool ok = row < n;
  for (int i0 = 0; i0 < per; i0 += 8) {   // (the same trips in every lane: the prefix sums run on whole waves)
    const int i = i0 + threadIdx.x / 32, h = hk * per + min(i, per - 1);
    const float dt = fmaxf(softplus_rule((float)a.a[(int64_t)rv * a.ab_stride + h] + a.dt_bias[h]), a.dt_min);
    double cum = ok ? (double)(dt * a.A[h]) : 0.0;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
      const double up = __shfl_up(cum, o, 32);
      if (row >= o) cum += up;
    }
    const double total = __shfl(cum, 31, 32);   // rows past the chunk's end add nothing
    if (i < per) {
      float* vec = ws + a.Hk * RC * RC + h * NV_SSM;
      const float hi = (float)cum;
      vec[row] = ok ? dt : 0.f;
      vec[RC + row] = hi;
      vec[2 * RC + row] = (float)(cum - (double)hi);
      vec[3 * RC + row] = ok ? __expf(hi) : 0.f;
      vec[4 * RC + row] = ok ? __expf((float)(total - cum)) : 0.f;
      if (row == 0) vec[5 * RC] = __expf((float)total);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The chunks of one (sequence, head) in order; block = NW waves x 16 value columns.  D rows of a 16 x 16
// product sit at 4 g + e, so with block b of S standing for key channels 32 (b / 2) + 8 (row / 4) + 4 (b % 2) +
// row % 4, blocks 2 s and 2 s + 1 of a lane are the eight k-slots of step s of k S and q S: S never
// leaves its registers.  S += k^T U takes k transposed out of the same LDS image (ds_read_b64_tr_b16).  The
// next chunk's rows and matrices travel to registers while this chunk is computed and to the other LDS
// buffer after it: one barrier per chunk.
// ---------------------------------------------------------------------------------------------
template <int DK>
__device__ __forceinline__ int img(int row, int chunk) { return row * (DK / 8) + (chunk ^ (row & (DK / 8 - 1))); }

__device__ __forceinline__ bf16x4 tr4(const bf16* base, int elem) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (s16x4 __attribute__((address_space(3)))*)((__attribute__((address_space(3))) bf16*)base + elem));
  return __builtin_bit_cast(bf16x4, v);
}

template <int DK, bool DELTA, int NW>
__global__ __launch_bounds__(64 * NW, 2) void chunk_rule_kernel(RuleArgs a) {
  constexpr int NS = DK / 32, NB = DK / 16, NT = 64 * NW;
  constexpr int NKL = RC * DK / 8 / NT, NML = RC * RC / 4 / NT;   // 16-byte loads per thread: k (and q), P (and T)
  static_assert(NKL * NT * 8 == RC * DK && NML * NT * 4 == RC * RC, "whole loads");
  __shared__ __attribute__((aligned(16))) bf16 sK[2][RC * DK], sQ[2][RC * DK];
  __shared__ __attribute__((aligned(16))) float sP[2][RC * LDM], sT[DELTA ? 2 : 1][DELTA ? RC * LDM : 4], sV[2][vec_floats<DELTA>()];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int s = blockIdx.z, h = blockIdx.x, hk = h / (a.H / a.Hk);
  const int n0 = (blockIdx.y * NW + (tid >> 6)) * 16;   // this wave's columns
  const bool live = n0 < a.dv;                          // dv is a multiple of 16: a wave has all of them or none
  const int r0 = a.cu[s], r1 = a.cu[s + 1];
  if (r1 <= r0) return;                                 // whole block
  const int chunks = (r1 - r0 + RC - 1) / RC;
  const int nc = (live ? n0 : 0) + col;

  // byte offsets of this thread's pieces within a chunk's 32 rows, against uniform bases; a last chunk of fewer
  // rows repeats its last one (whose scalars are zero)
  uint32_t ko[NKL], vo[8];
  auto offsets = [&](int n) {
#pragma unroll
    for (int i = 0; i < NKL; ++i) {
      const int e = tid + NT * i;
      ko[i] = 2 * ((uint32_t)min(e / (DK / 8), n - 1) * (uint32_t)a.stride + 8 * (e % (DK / 8)));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      vo[e] = 2 * ((uint32_t)min(16 * (e >> 2) + 4 * g + (e & 3), n - 1) * (uint32_t)a.v_stride + (uint32_t)nc);
  };
  const char* kp = reinterpret_cast<const char*>(a.k + (int64_t)r0 * a.stride + hk * DK);
  const char* qp = reinterpret_cast<const char*>(a.q + (int64_t)r0 * a.stride + hk * DK);
  const char* vp = reinterpret_cast<const char*>(a.v + (int64_t)r0 * a.v_stride + (int64_t)h * a.dv);
  const int64_t ws_step = 4 * ws_floats<DELTA>(a.H, a.Hk);
  const char* mp = reinterpret_cast<const char*>(a.ws) + (r0 / RC + s) * ws_step +
                   4 * (DELTA ? (int64_t)h * (2 * RC * RC + NV_DELTA) : (int64_t)hk * RC * RC);
  const uint32_t vec_at = 4 * (DELTA ? 2 * RC * RC : (a.Hk - hk) * RC * RC + h * NV_SSM);   // the vectors, from there
  bf16x8 rk[NKL], rq[NKL];
  f32x4 rp[NML], rt[NML], rvec, rhj[NML], rlj[NML];
  float rhi[NML], rli[NML];
  bf16 rv[8];
  auto fetch = [&](int c) {   // rows and matrices of chunk c
    if (r0 + (c + 1) * RC > r1) offsets(r1 - r0 - c * RC);
    const int64_t kc = (int64_t)c * RC * 2 * a.stride;
#pragma unroll
    for (int i = 0; i < NKL; ++i) {
      rk[i] = *reinterpret_cast<const bf16x8*>(kp + kc + ko[i]);
      rq[i] = *reinterpret_cast<const bf16x8*>(qp + kc + ko[i]);
    }
    const char* m = mp + c * ws_step;
#pragma unroll
    for (int i = 0; i < NML; ++i) {
      rp[i] = *reinterpret_cast<const f32x4*>(m + (uint32_t)(16 * (tid + NT * i)));
      if constexpr (DELTA) {
        rt[i] = *reinterpret_cast<const f32x4*>(m + (uint32_t)(4 * RC * RC + 16 * (tid + NT * i)));
      } else {
        const uint32_t e = tid + NT * i, hi = vec_at + 4 * (RC + e / (RC / 4)), hj = vec_at + 4 * (RC + 4 * (e % (RC / 4)));
        rhi[i] = *reinterpret_cast<const float*>(m + hi);
        rli[i] = *reinterpret_cast<const float*>(m + (hi + 4 * RC));
        rhj[i] = *reinterpret_cast<const f32x4*>(m + hj);
        rlj[i] = *reinterpret_cast<const f32x4*>(m + (hj + 4 * RC));
      }
    }
    if (tid < vec_floats<DELTA>() / 4) rvec = *reinterpret_cast<const f32x4*>(m + (vec_at + 16 * tid));
    const char* v = vp + (int64_t)c * RC * 2 * a.v_stride;
#pragma unroll
    for (int e = 0; e < 8; ++e) rv[e] = *reinterpret_cast<const bf16*>(v + vo[e]);
  };
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < NKL; ++i) {
      const int e = tid + NT * i, o = img<DK>(e / (DK / 8), e % (DK / 8)) * 8;
      st8(&sK[b][o], rk[i]);
      st8(&sQ[b][o], rq[i]);
    }
#pragma unroll
    for (int i = 0; i < NML; ++i) {
      const int e = tid + NT * i, row = e / (RC / 4), j = 4 * (e % (RC / 4)), o = row * LDM + j;
      if constexpr (!DELTA) {   // P_ij = q_i.k_j exp(cum_i - cum_j), j <= i; cum in two parts (long sums, short differences)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float p = rp[i][t] * __expf((rhi[i] - rhj[i][t]) + (rli[i] - rlj[i][t]));
          rp[i][t] = j + t <= row ? p : 0.f;
        }
      }
      *reinterpret_cast<f32x4*>(&sP[b][o]) = rp[i];
      if constexpr (DELTA) *reinterpret_cast<f32x4*>(&sT[b][o]) = rt[i];
    }
    if (tid < vec_floats<DELTA>() / 4) *reinterpret_cast<f32x4*>(&sV[b][4 * tid]) = rvec;
  };

  // state: lane (col, g) holds column nc, key channels 32 s + 8 g .. + 7 in blocks 2 s, 2 s + 1
  float* st = a.state + (((int64_t)a.slot[s] * a.H + h) * a.dv + nc) * DK + 8 * g;
  f32x4 S[NB];
  const auto start = [&] {
#pragma unroll
    for (int b = 0; b < NB; ++b)
      S[b] = a.reset[s] != 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(st + 32 * (b >> 1) + 4 * (b & 1));
  };
  start();
  const float Dh = DELTA ? 0.f : a.D[h];
  uint32_t oo[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) oo[e] = 2 * ((uint32_t)(16 * (e >> 2) + 4 * g + (e & 3)) * (uint32_t)a.out_stride + (uint32_t)nc);
  char* op = reinterpret_cast<char*>(a.out + (int64_t)r0 * a.out_stride + (int64_t)h * a.dv);

  // the sequence row by row, as the row-by-row kernels do it (each lane its 8 key channels of every 32)
  const auto walk = [&](int n) {
    for (int i = 0; i < n; ++i) {
      const int64_t row = r0 + i;
      bf16x8 k8[NS], q8[NS];
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        k8[t] = ld8(a.k + row * a.stride + hk * DK + 32 * t + 8 * g);
        q8[t] = ld8(a.q + row * a.stride + hk * DK + 32 * t + 8 * g);
      }
      const float x = (float)a.v[row * a.v_stride + (int64_t)h * a.dv + nc], ga = (float)a.a[row * a.ab_stride + h] + a.dt_bias[h];
      float decay, ik = 1.f, iq = 1.f, kq = 0.f, add;
      if constexpr (DELTA) {
        float nk = 0.f, nq = 0.f;
#pragma unroll
        for (int t = 0; t < NS; ++t)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            nk += (float)k8[t][j] * (float)k8[t][j];
            nq += (float)q8[t][j] * (float)q8[t][j];
            kq += (float)k8[t][j] * (float)q8[t][j];
          }
        ik = rsqrtf(group4_sum(nk) + 1e-6f);
        iq = rsqrtf(group4_sum(nq) + 1e-6f) * rsqrtf((float)DK);
        kq = group4_sum(kq) * ik * iq;
        decay = __expf(-__expf(a.A[h]) * softplus_rule(ga));
        float sk = 0.f;
#pragma unroll
        for (int t = 0; t < NS; ++t)
#pragma unroll
          for (int j = 0; j < 8; ++j) sk += S[2 * t + j / 4][j % 4] * ((float)k8[t][j] * ik);
        add = (x - decay * group4_sum(sk)) / (1.f + __expf(-(float)a.b[row * a.ab_stride + h]));
      } else {
        const float dt = fmaxf(softplus_rule(ga), a.dt_min);
        decay = __expf(dt * a.A[h]);
        add = dt * x;
      }
      float sq = 0.f;
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float s0 = S[2 * t + j / 4][j % 4], s1 = s0 * decay + (float)k8[t][j] * ik * add;
          sq += DELTA ? s0 * ((float)q8[t][j] * iq) : s1 * (float)q8[t][j];
          S[2 * t + j / 4][j % 4] = s1;
        }
      sq = group4_sum(sq);
      if (live && g == 0) a.out[row * a.out_stride + (int64_t)h * a.dv + nc] = (bf16)(DELTA ? decay * sq + add * kq : sq + Dh * x);
    }
  };

  const bool few = r1 - r0 <= FEW;                      // whole block
  bf16 vc[8];
  if (!few) {
    offsets(RC);
    fetch(0);
    put(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) vc[e] = rv[e];
    __syncthreads();
  }
  const auto step = [&](int c, int b) {
    if (c + 1 < chunks) fetch(c + 1);
    const bf16 *K = sK[b], *Q = sQ[b];
    // ---- k S and q S ----
    f32x4 ks[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      bf16x8 part[3], qa[2], ka[2];
      split3(S[2 * t], S[2 * t + 1], part);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int at = img<DK>(16 * rb + col, 4 * t + g) * 8;
        qa[rb] = ld8(&Q[at]);
        if constexpr (DELTA) ka[rb] = ld8(&K[at]);
      }
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          if constexpr (DELTA) ks[rb] = mma_bf16(ka[rb], part[p], ks[rb]);
          o[rb] = mma_bf16(qa[rb], part[p], o[rb]);
        }
    }
    // ---- R (DELTA) / U (Mamba-2) ----
    f32x4 r[2], u[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const f32x4 va = *reinterpret_cast<const f32x4*>(&sV[b][16 * rb + 4 * g]);
      const f32x4 vb = *reinterpret_cast<const f32x4*>(&sV[b][RC + 16 * rb + 4 * g]);
      const f32x4 vg = *reinterpret_cast<const f32x4*>(&sV[b][(DELTA ? 2 : 3) * RC + 16 * rb + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = (float)vc[4 * rb + e];
        r[rb][e] = va[e] * x;
        if constexpr (DELTA) r[rb][e] -= vb[e] * ks[rb][e];
        o[rb][e] = o[rb][e] * vg[e] + (DELTA ? 0.f : Dh * x);
      }
      u[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float gc = sV[b][(DELTA ? 4 : 5) * RC];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) S[nb] *= gc;
    // ---- U = T R, o += (P T) R (Mamba-2: o += P U) ----
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x4 pm[2], tm[2];
#pragma unroll
      for (int rb = kb; rb < 2; ++rb) {
        pm[rb] = *reinterpret_cast<const f32x4*>(&sP[b][(16 * rb + col) * LDM + 16 * kb + 4 * g]);
        if constexpr (DELTA) tm[rb] = *reinterpret_cast<const f32x4*>(&sT[b][(16 * rb + col) * LDM + 16 * kb + 4 * g]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int rb = kb; rb < 2; ++rb) {
          if constexpr (DELTA) u[rb] = mma_f32(tm[rb][e], r[kb][e], u[rb]);
          o[rb] = mma_f32(pm[rb][e], r[kb][e], o[rb]);
        }
    }
    // ---- S = g_C S + k^T U ----
    {
      bf16x8 part[3], ka[NB];
      const int qr = 4 * g + (col >> 2), p4 = col & 3;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int ch = 4 * (nb >> 1) + p4, half = 4 * (nb & 1);
        const bf16x4 lo = tr4(K, img<DK>(qr, ch) * 8 + half), hi = tr4(K, img<DK>(16 + qr, ch) * 8 + half);
        ka[nb] = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const f32x4 vd = *reinterpret_cast<const f32x4*>(&sV[b][(DELTA ? 3 : 4) * RC + 16 * rb + 4 * g]);
        u[rb] = (DELTA ? u[rb] : r[rb]) * vd;
      }
      split3(u[0], u[1], part);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) S[nb] = mma_bf16(ka[nb], part[p], S[nb]);
    }
    if (live) {
      char* oc = op + (int64_t)c * RC * 2 * a.out_stride;
      const int n = r1 - r0 - c * RC;
      if (n >= RC) {
#pragma unroll
        for (int e = 0; e < 8; ++e) *reinterpret_cast<bf16*>(oc + oo[e]) = (bf16)o[e >> 2][e & 3];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (16 * (e >> 2) + 4 * g + (e & 3) < n) *reinterpret_cast<bf16*>(oc + oo[e]) = (bf16)o[e >> 2][e & 3];
      }
    }
    if (c + 1 < chunks) {
      put(b ^ 1);   // last read before the previous barrier
#pragma unroll
      for (int e = 0; e < 8; ++e) vc[e] = rv[e];
    }
    __syncthreads();
  };
  for (int c = 0; !few && c < chunks; c += 2) {
    step(c, 0);
    if (c + 1 < chunks) step(c + 1, 1);
  }
  float broken = 0.f;   // NaN if a value of S is not finite
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int e = 0; e < 4; ++e) broken += S[nb][e] * 0.f;
  if (live && (few || __ballot(broken != 0.f))) {
    if (!few) start();
    walk(r1 - r0);
  }
  if (live) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) *reinterpret_cast<f32x4*>(st + 32 * (nb >> 1) + 4 * (nb & 1)) = S[nb];
  }
}

template <bool DELTA>
int launch_rule(const RuleArgs& a, int T, int dk, hipStream_t stream) {
  const dim3 gram(T / RC + a.S, DELTA ? (a.H + 3) / 4 : a.Hk);
  const dim3 rule(a.H, (a.dv + 63) / 64, a.S);
  if (dk == 128) {
    if constexpr (DELTA) chunk_gram_kernel<128><<<gram, 256, 0, stream>>>(a);
    else ssm_gram_kernel<128><<<gram, 256, 0, stream>>>(a);
    chunk_rule_kernel<128, DELTA, 4><<<rule, 256, 0, stream>>>(a);
  } else {
    if constexpr (DELTA) chunk_gram_kernel<64><<<gram, 256, 0, stream>>>(a);
    else ssm_gram_kernel<64><<<gram, 256, 0, stream>>>(a);
    chunk_rule_kernel<64, DELTA, 4><<<rule, 256, 0, stream>>>(a);
  }
  OME_CHECK_LAUNCH();
  return 0;
}

// (row strides below 2^24 elements: a chunk's byte offsets stay in 32 bits)
bool rule_shape(int S, int H, int Hk, int dk, int dv, int64_t s0, int64_t s1, int64_t s2) {
  return s0 >= 0 && s1 >= 0 && s2 >= 0 && s0 < 1 << 24 && s1 < 1 << 24 && s2 < 1 << 24 && S > 0 && S <= 65535 && H > 0 && Hk > 0 && H % Hk == 0 && (dk == 64 || dk == 128) && dv > 0 && dv % 16 == 0 &&
         (dv + 63) / 64 <= 65535 && H <= 65535;
}

bool aligned16(const void* p, int64_t elems) { return ((uintptr_t)p | (uintptr_t)(elems * 2)) % 16 == 0; }

}  // namespace

// fp32 words of workspace of one chunk of H heads (Mamba-2: in G groups); T rows of S sequences have up to T / 32 + S
OME_API int ome_chunk_rule_floats(int H, int G, int delta) {
  return (int)(delta ? ws_floats<true>(H, G) : ws_floats<false>(H, G));
}

// Gated delta rule over all rows of every sequence; operands as ome_gdn_scan.  -3: a shape, stride or
// alignment that the chunked kernels do not take (nothing is launched).
OME_API int ome_gdn_chunks(const void* q, const void* k, const void* v, int64_t qkv_stride, const void* a, const void* b,
                           int64_t ab_stride, const float* A_log, const float* dt_bias, float* state, void* out,
                           int64_t out_stride, const int* cu, const int* slot, const int* reset, int S, int T, int Hv, int Hk,
                           int dk, int dv, float* ws, hipStream_t stream) {
  if (T <= 0 || !ws || !rule_shape(S, Hv, Hk, dk, dv, qkv_stride, qkv_stride, out_stride) || !aligned16(q, qkv_stride) || !aligned16(k, qkv_stride) ||
      (uintptr_t)state % 16 || (uintptr_t)ws % 16)
    return -3;
  const RuleArgs r{(const bf16*)q, (const bf16*)k, (const bf16*)v, qkv_stride, qkv_stride, (const bf16*)a, (const bf16*)b,
                   ab_stride, A_log, nullptr, dt_bias, 0.f, ws, state, (bf16*)out, out_stride, cu, slot, reset, S, Hv, Hk, dv};
  return launch_rule<true>(r, T, dk, stream);
}

// Mamba-2's selective scan over all rows of every sequence; operands as ome_ssm_scan.
OME_API int ome_ssm_chunks(const void* x, int64_t x_stride, const void* dt, int64_t dt_stride, const void* B, const void* Cm,
                           int64_t bc_stride, const float* A, const float* D, const float* dt_bias, float dt_min, float* state,
                           void* y, int64_t y_stride, const int* cu, const int* slot, const int* reset, int S, int T, int H,
                           int P, int N, int G, float* ws, hipStream_t stream) {
  if (T <= 0 || !ws || !rule_shape(S, H, G, N, P, bc_stride, x_stride, y_stride) || !aligned16(B, bc_stride) || !aligned16(Cm, bc_stride) ||
      (uintptr_t)state % 16 || (uintptr_t)ws % 16)
    return -3;
  const RuleArgs r{(const bf16*)Cm, (const bf16*)B, (const bf16*)x, bc_stride, x_stride, (const bf16*)dt, nullptr,
                   dt_stride, A, D, dt_bias, dt_min, ws, state, (bf16*)y, y_stride, cu, slot, reset, S, H, G, P};
  return launch_rule<false>(r, T, N, stream);
}
