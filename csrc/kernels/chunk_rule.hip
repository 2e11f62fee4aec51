// Prompt rows of the matrix-state layers with one decay per head, in chunks of 32 rows on the matrix
// cores (gfx950): the gated delta rule of Qwen3-Next / Jet-Nemotron (DELTA) and the selective scan of
// Mamba-2 (not DELTA).  With S [dk, dv] the state a chunk starts from, k_i / q_i its key and query
// rows (unit-norm for DELTA, B / C for Mamba-2), g_i = exp(cum_i) the decay from the chunk's start up to and
// with row i:
//   DELTA   A_ij = beta_i exp(cum_i - cum_j) k_i.k_j (j < i),  T = (I + A)^-1,
//           U = T R,  R_i = beta_i (v_i - g_i k_i S)                    Mamba-2   U_i = dt_i x_i (P's columns and the last
//                                                                            factors below take dt_i: x_i stays as it is)
//   o_i = g_i q_i S + sum_{j <= i} P_ij U_j,  P_ij = exp(cum_i - cum_j) q_i.k_j     (+ D x_i)
//       (DELTA: P U = (P T) R, so that o and U both follow from R)
//   S'  = g_C S + sum_i exp(cum_C - cum_i) k_i U_i^T
//
// Two launches.  chunk_gram_kernel (Mamba-2: ssm_gram_kernel), parallel over all rows: the 32 x 32 matrices
// P T and T (Mamba-2: q k^T, which the heads of a group share) and the chunk's scalars, into a workspace.
// chunk_rule_kernel walks the chunks of a (sequence, head) in order: a wave owns 16 value columns and keeps its
// S in VGPR accumulators.  Long prompts of few heads are cut into segments that are walked side by side, in two launches of it
// (ops._chunk_rule_seg; S at a segment's end is linear in S at its start): whole layers of one prompt of 8000 rows, 8 heads of 128 x 128
// 489 -> 195 us, 32 heads of 64 x 128 435 -> 158.  The state's error against 64 bits, eight prompts of 1000 to 8000 rows: 1.10e-7 both ways (8.55e-8).
//
// What bounds it: the instructions of a wave that has its SIMD almost for itself, 96 matrix (Mamba-2: 54) and some 250 (270) vector
// ones a chunk.  A product takes 16 cycles alone, but about 9 of them stay its own where vector instructions of 4 cycles fill
// the rest, so a chunk is 2000 cycles of issue and some 1400 of LDS latency and dependencies.  Hence the
// next chunk moves to LDS by DMA, without a register or a store on the way, and where a workgroup has its CU to itself by two waves of their own: a
// move holds its wave up for some 50 cycles, and the nine of a wave that also computes took a quarter of its time (scan of a delta rule, 192
// workgroups 91 -> 73 us, now 70, 64 61 -> 49, now 47; selective scan, 256 54 -> 43, now 42, 128 40 -> 32, now 31; moves by one or by four such waves 73 and 77 for the first).  With two
// workgroups a CU each covers the other's moves, and such waves only take slots from them (448 workgroups 36.7 -> 37.8, 512 76 -> 81): none there.  Values and outputs move in pieces of four columns
// (q S is formed transposed for that); T and P T are products of three bf16 parts each, at half the fp32 product's time.
// Memory traffic hides behind that.  Two fp16 parts instead of three bf16 ones would take a quarter less time, but the state came out
// 2.3 times further from 64 bits: an fp16 value below 2^-14 has no lower part.
// (chunks' matrices + scan, calls that are waited for one by one):
//   gated delta rule, 32 heads of 128 x 128, prompts of 1001 / 1435 / 1564 rows:   20 + 70 us (before: 24 + 123; row by row: 1098)
//   selective scan, 128 heads of 64 x 128, 8 groups, 1033 / 926 / 1248 / 293 rows:  9 + 74 us (values scaled by dt in three parts: 10 + 93; before: 11 + 116;
//   row by row: 1745)
// Largest error of the state against 64 bits: 1.2e-7 (row by row: 2.0e-7) and 1.2e-7 (6.2e-7) of its norm.
//
// A chunk's products multiply the entries that causality zeroes as well, and 0 times an infinity or NaN is NaN, so a key,
// gate or value that is not finite would reach the rows before it in its chunk.  It reaches S and stays there (each
// U_i enters every channel of S, and no decay takes an infinity or NaN away), so S tells at the end of a sequence: a
// wave whose S is not finite walks its columns again row by row.
//
// fp32 throughout: k and q enter the matrix cores as the bf16 values that they are (their norms, 1 / |k| and
// 1 / (|q| sqrt(dk)), scale results), S and U as three bf16 parts that sum to the fp32 value exactly, at
// 3/16 of the fp32 MFMA's time; T R and P T R, where both operands are fp32, take the six products of their parts down to
// 2^-16 of the first (what is left out is below 2^-24, an fp32 rounding).  Decay exponents are summed in fp64 (differences of
// a long sum).  The row-by-row kernels stay for decode steps (one row per sequence), few rows in all, dk other than 64 / 128, and
// unaligned views of q and k.
#include "common.h"

namespace {

constexpr int RC = 32;            // rows of a chunk
constexpr int LDM = RC + 4;       // padded row of a 32 x 32 fp32 matrix in LDS
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Workspace of one chunk, in bytes: (Mamba-2) of every group q k^T in fp32, which its heads share (they differ in their decays only,
// which the scan applies: P itself would be 16 times the bytes); of every head (DELTA) the images of T and P T, each in three
// bf16 parts, as LDS holds them, and its vectors, 32 floats each: DELTA a, b, c, d of the scan, then g_C;  Mamba-2 dt, pairs of cum's upper and
// lower part (of two to the power), c, d, P's diagonal, then g_C.
constexpr int MAT = RC * RC * 2;      // a part of a 32 x 32 matrix
constexpr int VECS = 1024;            // the vectors, in whole LDS moves
template <bool DELTA>
constexpr int vec_floats() { return (DELTA ? 4 : 6) * RC + 4; }
template <bool DELTA>
__host__ __device__ constexpr int64_t group_bytes() { return DELTA ? 0 : 4 * RC * RC; }
template <bool DELTA>
__host__ __device__ constexpr int64_t head_bytes() { return (DELTA ? 6 * MAT : 0) + VECS; }
template <bool DELTA>
__host__ __device__ constexpr int64_t ws_bytes(int H, int G) { return G * group_bytes<DELTA>() + H * head_bytes<DELTA>(); }

struct RuleArgs {
  const bf16 *q, *k, *v;          // rows of stride `stride` (v: v_stride)
  int64_t stride, v_stride;
  const bf16 *a, *b;              // per-head rows: a | b (DELTA), dt (Mamba-2)
  int64_t ab_stride;
  const float *A, *D, *dt_bias;   // A_log (DELTA) / A, D (Mamba-2)
  float dt_min;
  char* ws;
  float* state;                   // [slots, H, dv, dk]
  bf16* out;
  int64_t out_stride;
  const int *cu, *slot, *reset;
  int S, H, Hk, dv;
  int seg;                        // chunks of a segment (0: sequences in one piece)
  float* segs;                    // seg_floats of every (segment, head)
  int4* turn;                     // the sequences in the order of their workgroups (set_turns), or null: as they come
};

constexpr int TURNS = 64;         // of at most so many

// A sequence: its number, rows, place in the state, whether it starts afresh.
struct Seq {
  int s, q0, q1, slot;
  bool fresh;
};

__device__ __forceinline__ Seq seq_of(const RuleArgs& a, int s) { return {s, a.cu[s], a.cu[s + 1], a.slot[s], a.reset[s] != 0}; }

// The order of the sequences' workgroups: the longest first, and of the sequences that begin a second round over the CUs
// the shortest first, so that a CU's two workgroups are as long as another's (four prompts of 293 to 1248 rows, 128 heads: 106 -> 93 us).
// Set beside the chunks' matrices, by the last workgroup, which rarely has a chunk; a workgroup of the scan then reads a sequence whole.
// (Searched by each workgroup of the scan it took as long as a short sequence.  10 prompts of 33 rows beside 50 of 1, delta rule of 32 heads
// and selective scan of 128: 74 and 113 us so, 54 and 75 now and without an order; 48 prompts of 30 to 289 rows 204 and 293 -> 190 and 279.)
__device__ __forceinline__ void set_turns(const RuleArgs& a) {
  if (a.turn == nullptr || blockIdx.x != gridDim.x - 1 || blockIdx.y != 0 || threadIdx.x >= 64) return;
  const int lane = threadIdx.x, len = lane < a.S ? a.cu[lane + 1] - a.cu[lane] : -1;
  const Seq own = seq_of(a, min(lane, a.S - 1));
  int rank = 0;
  for (int j = 0; j < a.S; ++j) {
    const int other = __builtin_amdgcn_readlane(len, j);
    rank += other > len || (other == len && j < lane);
  }
  const int round = max(256 / (a.H * ((a.dv + 63) / 64)), 1), k = rank / round;
  if (lane < a.S) a.turn[k & 1 ? min(a.S, (k + 1) * round) - 1 - (rank - k * round) : rank] = int4{own.s | (own.fresh ? 1 << 31 : 0), own.q0, own.q1, own.slot};
}

// Floats that a segment leaves of a head: its state [dv, dk]; then DELTA its transition [dk, dk], Mamba-2 its decay (a sequence's first
// segment: what the sequence started from).
__host__ __device__ constexpr int64_t seg_floats(int dv, int dk) { return (int64_t)dv * dk + (int64_t)(dv > dk ? dv : dk) * dk + 4; }

// Segment `id` of `R` rows -> (sequence, number in it); ids as those of chunks below.  Whole wave.
__device__ __forceinline__ bool segment_of(int id, int R, const int* cu, int S, int& s, int& j) {
  const int lane = threadIdx.x & 63;
  s = -1;
  for (int b = 0; b < S; b += 64) {
    const int i = b + lane;
    const int c = __popcll(__ballot(i < S && cu[min(i, S)] / R + i <= id));
    s += c;
    if (c < 64) break;
  }
  s = __builtin_amdgcn_readfirstlane(s);
  if (s < 0) return false;
  j = id - cu[s] / R - s;
  return cu[s] + (int64_t)j * R < cu[s + 1];
}

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

// Eight fp32 values -> three bf16 vectors that sum to them exactly.  What a rounding took by v_dot2_f32_bf16, the value minus the
// half of a packed pair: seven instructions a pair (eleven by masks, shifts and subtractions).
__device__ __forceinline__ void split3(f32x4 x0, f32x4 x1, bf16x8 (&p)[3]) {
  uint32_t lo = 0x0000bf80u, hi = 0xbf800000u;   // (-1, 0) and (0, -1); out of sight, or they become inline constants, of which
  asm("" : "+s"(lo), "+s"(hi));                  // the instruction takes another pair of halves
  const bf16x2 first = __builtin_bit_cast(bf16x2, lo), second = __builtin_bit_cast(bf16x2, hi);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = j < 2 ? x0[2 * j] : x1[2 * j - 4], b = j < 2 ? x0[2 * j + 1] : x1[2 * j - 3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const bf16x2 h = {(bf16)a, (bf16)b};
      p[t][2 * j] = h[0];
      p[t][2 * j + 1] = h[1];
      if (t < 2) {
        a = __builtin_amdgcn_fdot2_f32_bf16(h, first, a, false);
        b = __builtin_amdgcn_fdot2_f32_bf16(h, second, b, false);
      }
    }
  }
}

// Two, by cutting the lower bits off: half as many instructions again, but a dot product waits for the products around it (20 cycles each way).
// For a wave that has little else to do beside its products (Mamba-2's P: 2% of the scan; S and U so: 1 to 2% more).
__device__ __forceinline__ void cut3(float a, float b, uint32_t (&p)[3]) {
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const uint32_t u = __float_as_uint(a), v = __float_as_uint(b);
    p[t] = __builtin_amdgcn_perm(v, u, 0x07060302u);
    a -= __uint_as_float(u & 0xffff0000u);
    b -= __uint_as_float(v & 0xffff0000u);
  }
}

// c + a b of operands in three parts: the six products down to 2^-16 of the first
template <bool SWAP = false>
__device__ __forceinline__ void mma_parts(const bf16x8 (&a)[2][3], const bf16x8 (&b)[3], f32x4 (&c)[2]) {
#pragma unroll
  for (int sum = 2; sum >= 0; --sum)
#pragma unroll
    for (int i = 0; i <= sum; ++i)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) c[rb] = SWAP ? mma_bf16(b[sum - i], a[rb][i], c[rb]) : mma_bf16(a[rb][i], b[sum - i], c[rb]);
}

// LDS written by lanes of a wave, read by others of the same wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float softplus_rule(float x) { return x > 20.f ? x : log1pf(__expf(x)); }

// 16-byte piece `chunk` of row `row` in an image of k or q rows; byte offset of columns 4 g .. + 3 and 16 + 4 g .. + 3 (the
// k-slots of a lane of group g) of row `row` in a part of a 32 x 32 matrix; piece of eight columns in an image of values.
// Swizzled, so that the pieces of 16 rows (k and q: and four pieces of four rows, as a transposed read takes them) lie in all banks.
template <int DK>
__device__ __forceinline__ int img(int row, int chunk) {
  return row * (DK / 8) + (chunk ^ (DK == 128 ? (row & 3) << 2 | ((row >> 2) & 3) : ((row >> 1) & 1) << 2 | ((row >> 2) & 3)));
}
__device__ __forceinline__ int mat_img(int row, int g) { return row * (RC * 2) + ((g ^ ((row >> 2) & 3)) << 4); }
__device__ __forceinline__ int val_img(int row, int piece) { return row * 8 + (piece ^ (((row >> 1) & 3) << 1)); }

__device__ __forceinline__ bf16x4 tr4(const bf16* base, int elem) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (s16x4 __attribute__((address_space(3)))*)((__attribute__((address_space(3))) bf16*)base + elem));
  return __builtin_bit_cast(bf16x4, v);
}

// ---------------------------------------------------------------------------------------------
// One wave per (chunk, head).  The 16-byte row pieces that a lane loads are both operands of q k^T and
// k k^T (rows and columns of a 16 x 16 x 32 product have the same lane layout).  T's diagonal blocks by forward substitution:
// lane j keeps column j in registers and reads the rows of A from LDS as broadcasts.
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
  set_turns(a);
  if (h >= a.H || !chunk_of(blockIdx.x, a.cu, a.S, r0, n)) return;   // whole wave; no block barrier below
  const int hk = h / (a.H / a.Hk);
  char* ws = a.ws + blockIdx.x * ws_bytes<true>(a.H, a.Hk) + h * head_bytes<true>();

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
    float* vec = reinterpret_cast<float*>(ws + 6 * MAT);
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
  // T in blocks of 16: T11 and T22 by substitution, in place of A11 and A22; T21 = -T22 (A21 T11)
  const int d16 = row & 16;
  float t[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float acc[4] = {i == col ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < i; m += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&sA[w][(d16 + i) * LDM + d16 + m]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (m + e < i) acc[e] -= x[e] * t[m + e];
    }
    t[i] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < 16; ++i) sA[w][(d16 + i) * LDM + d16 + col] = t[i];   // (both half waves the same)
  wave_sync();
  // operands of 16 x 16 x 4 products: the k-slot of step e is row (column) 4 g + e
  f32x4 tb[2][2];   // T [row block][column block], as a right operand
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) tb[d][d][e] = sA[w][(16 * d + 4 * g + e) * LDM + 16 * d + col];
  const f32x4 a21 = *reinterpret_cast<const f32x4*>(&sA[w][(16 + col) * LDM + 4 * g]), t22 = *reinterpret_cast<const f32x4*>(&sA[w][(16 + col) * LDM + 16 + 4 * g]);
  f32x4 at = {0.f, 0.f, 0.f, 0.f};
  tb[1][0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e) at = mma_f32(-a21[e], tb[0][0][e], at);
#pragma unroll
  for (int e = 0; e < 4; ++e) tb[1][0] = mma_f32(t22[e], at[e], tb[1][0]);
  wave_sync();
#pragma unroll
  for (int e = 0; e < 4; ++e) sA[w][(16 + 4 * g + e) * LDM + col] = tb[1][0][e];
  wave_sync();
  // a 32 x 32 matrix out of LDS, in three bf16 parts, to its images
  const auto parts = [&](char* to) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(&sA[w][(16 * rb + col) * LDM + 4 * g]);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(&sA[w][(16 * rb + col) * LDM + 16 + 4 * g]);
      bf16x8 p[3];
      split3(lo, hi, p);
#pragma unroll
      for (int x = 0; x < 3; ++x) *reinterpret_cast<bf16x8*>(to + x * MAT + mat_img(16 * rb + col, g)) = p[x];
    }
  };
  parts(ws);
  wave_sync();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb <= rb; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) sA[w][(16 * rb + 4 * g + e) * LDM + 16 * cb + col] = pm[rb][cb][e];
  wave_sync();
  f32x4 pt[2][2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      pt[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = cb; kb <= rb; ++kb) {
        const f32x4 m = *reinterpret_cast<const f32x4*>(&sA[w][(16 * rb + col) * LDM + 16 * kb + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) pt[rb][cb] = mma_f32(m[e], tb[kb][cb][e], pt[rb][cb]);
      }
    }
  wave_sync();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) sA[w][(16 * rb + 4 * g + e) * LDM + 16 * cb + col] = pt[rb][cb][e];
  wave_sync();
  parts(ws + 3 * MAT);
}

// Mamba-2: one block per (chunk, group).  Wave 0 multiplies q k^T (lower triangle), every half wave takes heads.
template <int DK>
__global__ __launch_bounds__(256) void ssm_gram_kernel(RuleArgs a) {
  constexpr int NS = DK / 32;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, hk = blockIdx.y;
  int r0, n;
  set_turns(a);
  if (!chunk_of(blockIdx.x, a.cu, a.S, r0, n)) return;   // the same in every wave
  char* ws = a.ws + blockIdx.x * ws_bytes<false>(a.H, a.Hk);
  __shared__ float s_diag[RC];
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
    float* gram = reinterpret_cast<float*>(ws + hk * group_bytes<false>());
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb <= rb; ++cb) {
        f32x4 qk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s) qk = mma_bf16(qf[rb][s], kf[cb][s], qk);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          gram[(16 * rb + 4 * g + e) * RC + 16 * cb + col] = qk[e];
          if (cb == rb && 4 * g + e == col) s_diag[16 * rb + col] = qk[e];
        }
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
    float* vec = reinterpret_cast<float*>(ws + a.Hk * group_bytes<false>() + h * head_bytes<false>());
    if (i < per) {
      const double two = cum * 1.4426950408889634;
      const float hi = (float)two;
      vec[row] = ok ? dt : 0.f;
      *reinterpret_cast<float2*>(vec + RC + 2 * row) = float2{hi, (float)(two - (double)hi)};
      vec[3 * RC + row] = ok ? __expf((float)cum) : 0.f;
      vec[4 * RC + row] = ok ? dt * __expf((float)(total - cum)) : 0.f;
      if (row == 0) vec[6 * RC] = __expf((float)total);
    }
    if (i0 == 0) __syncthreads();   // (s_diag)
    if (i < per) vec[5 * RC + row] = ok ? dt * s_diag[row] : 0.f;
  }
}

// ---------------------------------------------------------------------------------------------
// The chunks of one (sequence, head) in order; block = NW waves x 16 value columns.  D rows of a 16 x 16
// product sit at 4 g + e, so with block b of S standing for key channels 32 (b / 2) + 8 (row / 4) + 4 (b % 2) +
// row % 4, blocks 2 s and 2 s + 1 of a lane are the eight k-slots of step s of k S and q S: S never
// leaves its registers.  S += k^T U takes k transposed out of the same LDS image (ds_read_b64_tr_b16).  The
// next chunk moves to the other LDS buffer while this one is computed: one barrier per chunk.  MW > 0: by MW further waves, which do
// nothing else and meet the others at each of their barriers; 0: by the waves that compute.
// VEC: values in 16-byte pieces by DMA, outputs in 8-byte ones; not: element by element (views that are not aligned for that).
//
// SEG: few sequences of few heads leave most of the chip idle for their length, so they run in segments side by side.
//   1  a segment's own state: S from zero (a sequence's first segment: from where the sequence starts), without outputs, and for DELTA its
//      transition M, the state of the identity's columns without values (workgroups beyond the values' in y).  The last segment has none.
//   2  the segment itself, from S = M_i S + S_i over the segments before it (Mamba-2: M is the product of the decays).
// ---------------------------------------------------------------------------------------------
template <int DK, bool DELTA, int NW, bool VEC, int SEG, int MW>
__global__ __launch_bounds__(64 * (NW + MW), 2) void chunk_rule_kernel(RuleArgs a) {
  constexpr int NS = DK / 32, NB = DK / 16, NT = 64 * NW, COLS = 16 * NW;
  static_assert(RC * COLS == 8 * NT && RC * RC / 4 == NT, "whole loads; a pair below P's diagonal a thread");
  // a chunk in LDS: k and q rows, T and P T (Mamba-2: P) in three parts each, the vectors, the values
  constexpr int ROWS = RC * DK * 2, M_AT = 2 * ROWS, V_AT = M_AT + (DELTA ? 6 : 3) * MAT, X_AT = V_AT + VECS, IMG = X_AT + RC * COLS * 2;
  __shared__ __attribute__((aligned(1024))) char lds[2 * IMG];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)lds;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15, g = lane >> 4;
  int j = 0;
  Seq seq;
  if constexpr (SEG == 0) {
    if (a.turn != nullptr) {
      const int4 t = a.turn[blockIdx.z];
      seq = {t.x & 0x7fffffff, t.y, t.z, t.w, t.x < 0};
    } else {
      seq = seq_of(a, blockIdx.z);
    }
  } else {
    int id;
    if (!segment_of(blockIdx.z, a.seg * RC, a.cu, a.S, id, j)) return;
    seq = seq_of(a, id);
  }
  const int s = seq.s, h = blockIdx.x, hk = h / (a.H / a.Hk);
  const int q0 = seq.q0, r0 = q0 + j * a.seg * RC, r1 = SEG ? min(seq.q1, r0 + a.seg * RC) : seq.q1;
  if (r1 <= r0) return;                                    // whole block
  const bool last = SEG == 0 || r1 == seq.q1;
  const bool ident = SEG == 1 && DELTA && blockIdx.y >= (a.dv + COLS - 1) / COLS;   // columns of the transition
  if (SEG == 1 && (last || (ident && j == 0))) return;
  const int c0 = (ident ? blockIdx.y - (a.dv + COLS - 1) / COLS : blockIdx.y) * COLS, n0 = c0 + wave * 16;   // the block's and this wave's columns
  const bool live = ident || n0 < a.dv;                    // dv is a multiple of 16: a wave has all of them or none
  float* const sg = SEG ? a.segs + ((int64_t)blockIdx.z * a.H + h) * seg_floats(a.dv, DK) : nullptr;   // this segment's
  const int64_t sg_step = (int64_t)a.H * seg_floats(a.dv, DK);
  const int chunks = (r1 - r0 + RC - 1) / RC;
  const int nc = (live ? n0 : 0) + col;

  const bool few = r1 - r0 <= FEW && j == 0;            // whole block
  // The moves of a chunk to LDS are cut into NW shares; a wave that moves has K of them: w0, w0 + MW, ...
  constexpr int K = MW ? NW / MW : 1, KS = MW ? MW : NW;
  static_assert(K * KS == NW && COLS == 64 && NT * 4 == VECS, "whole shares; eight pieces a row of values; a float a thread");
  const int w0 = MW ? wave - NW : wave;
  // values: a lane's row and eight columns (beyond dv: the first eight); a last chunk of fewer rows repeats its last one (whose scalars are zero)
  // rows of k and q: a lane's 16-byte piece of each move of 1024 bytes, against uniform bases
  constexpr int NR = ROWS / 1024 / NW, NH = (int)head_bytes<DELTA>() / 1024;
  static_assert(NR * NW * 1024 == ROWS && (NH - 1) % NW == 0, "whole moves");
  uint32_t xo[K], ko[K][NR];
  const auto offsets = [&](int n) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int vt = 64 * (w0 + KS * k) + lane, xr = vt / 8, xp8 = 8 * (val_img(xr, vt % 8) - 8 * xr), xc = c0 + xp8 < a.dv ? xp8 : 0;
      xo[k] = 2 * ((uint32_t)min(xr, n - 1) * (uint32_t)a.v_stride + (uint32_t)xc);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int e = 64 * (w0 + KS * k + NW * i) + lane, row = e / (DK / 8);
        ko[k][i] = 2 * ((uint32_t)min(row, n - 1) * (uint32_t)a.stride + 8 * (uint32_t)(img<DK>(row, e % (DK / 8)) - row * (DK / 8)));
      }
    }
  };
  const int64_t x_step = (int64_t)RC * 2 * a.v_stride, k_step = (int64_t)RC * 2 * a.stride, ws_step = ws_bytes<DELTA>(a.H, a.Hk);
  const char* xp = reinterpret_cast<const char*>(a.v + (int64_t)r0 * a.v_stride + (int64_t)h * a.dv + c0);   // these walk with the chunks moved
  const char* kp = reinterpret_cast<const char*>(a.k + (int64_t)r0 * a.stride + hk * DK);
  const char* qp = reinterpret_cast<const char*>(a.q + (int64_t)r0 * a.stride + hk * DK);
  const char* gp = a.ws + (q0 / RC + s + j * a.seg) * ws_step + hk * group_bytes<DELTA>();
  const char* hp = a.ws + (q0 / RC + s + j * a.seg) * ws_step + a.Hk * group_bytes<DELTA>() + h * head_bytes<DELTA>();
  // A chunk of n rows to LDS buffer b.  `more`: there is one; without, nothing is moved (no branch, which would part a step's stages).
  const auto move = [&](int n, bool more, int b) __attribute__((always_inline)) {
    if (more && n < RC) offsets(n);
    const uint32_t to = lds0 + b * IMG, kb = (RC - 1) * 2 * (uint32_t)a.stride + 2 * DK;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int w = w0 + KS * k;
      if constexpr (VEC) buffer_to_lds(xp, more && !ident ? (uint32_t)(RC - 1) * 2 * (uint32_t)a.v_stride + 2 * COLS : 0, xo[k], 0, to + X_AT + 1024 * w);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        buffer_to_lds(kp, more ? kb : 0, ko[k][i], 0, to + 1024 * (w + NW * i));
        if constexpr (SEG != 1) buffer_to_lds(qp, more ? kb : 0, ko[k][i], 0, to + ROWS + 1024 * (w + NW * i));
      }
#pragma unroll
      for (int i = 0; i < (NH - 1) / NW; ++i) buffer_to_lds(hp, more ? (NH - 1) * 1024 : 0, 16 * lane, 1024 * (w + NW * i), to + M_AT + 1024 * (w + NW * i));
      buffer_to_lds4(hp + (NH - 1) * 1024, more ? 4 * vec_floats<DELTA>() : 0, 4 * (64 * w + lane), to + V_AT + 256 * w);
    }
  };
  const auto advance = [&](bool more) __attribute__((always_inline)) {
    xp += more ? x_step : 0;
    kp += more ? k_step : 0;
    qp += more ? k_step : 0;
    gp += more ? ws_step : 0;
    hp += more ? ws_step : 0;
  };
  if (MW && wave >= NW) {
    if (few) return;
    if constexpr (SEG == 2 && DELTA) {   // the barriers of `start`
      for (int i = 1; i < j; ++i) {
        if (i > 1) __syncthreads();
        __syncthreads();
      }
      if (j > 1) __syncthreads();
    }
    offsets(RC);
    for (int c = 0; c < chunks; ++c) {   // (the buffer was read last before the previous barrier)
      move(r1 - r0 - c * RC, true, c & 1);
      advance(true);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    __syncthreads();
    return;
  }

  // What goes through registers comes a chunk ahead of the products: q k^T and its decays (Mamba-2), values by element.  Without a next chunk
  // it is the last one again (no branch, which would part the stages).
  // Mamba-2: a thread forms two neighbours of P below its diagonal, which itself joins D.  (Four of all 1024 values, of which half are zero: twice the vector
  // instructions, some 60 of a chunk's 430; scan of 128 workgroups 32.0 -> 30.6 us, 256 42.8 -> 41.6, 512 76.7 -> 75.2.)  Rows 2 m - 1 and 2 m have m pairs each (row 31: 16), so 32 threads take the rows of m and of 16 - m.
  int prow = 31, pcol = 2 * (tid % 16);
  {
    const int m = tid / 32 + 1, i = tid % 32, n = i < 2 * m ? m : 16 - m, k = i < 2 * m ? i : i - 2 * m;
    if (m < 8 || i < 16) prow = 2 * n - 1 + (k >= n), pcol = 2 * (k >= n ? k - n : k);
  }
  f32x2 rp, rdj;
  f32x4 rcj;
  f32x2 rci;
  bf16x8 rx;
  const auto ahead = [&](int c) __attribute__((always_inline)) {   // of chunk c
    if constexpr (!VEC) {
      const int xr = min(tid / 8, r1 - r0 - c * RC - 1), xp8 = 8 * (val_img(tid / 8, tid % 8) - 8 * (tid / 8));
      const bf16* x = a.v + (int64_t)(r0 + c * RC + xr) * a.v_stride + (int64_t)h * a.dv + c0 + (c0 + xp8 < a.dv ? xp8 : 0);
#pragma unroll
      for (int e = 0; e < 8; ++e) rx[e] = x[e];
    }
    if constexpr (!DELTA && SEG != 1) {
      rp = *reinterpret_cast<const f32x2*>(gp + (uint32_t)(4 * (prow * RC + pcol)));
      rdj = *reinterpret_cast<const f32x2*>(hp + (uint32_t)(4 * pcol));
      rcj = *reinterpret_cast<const f32x4*>(hp + (uint32_t)(4 * (RC + 2 * pcol)));
      rci = *reinterpret_cast<const f32x2*>(hp + (uint32_t)(4 * (RC + 2 * prow)));
    }
  };
  const auto pair_at = [](int row, int c) { return mat_img(row, (c & 15) >> 2) + 8 * (c >> 4) + 2 * (c & 3); };
  const auto put = [&](int b) __attribute__((always_inline)) {   // P_ij dt_j = q_i.k_j exp(cum_i - cum_j) dt_j, j < i; cum in two parts (long sums, short differences)
    if constexpr (!VEC) *reinterpret_cast<bf16x8*>(lds + b * IMG + X_AT + 16 * tid) = rx;
    if constexpr (!DELTA && SEG != 1) {
      const float x0 = rp[0] * __builtin_amdgcn_exp2f((rci[0] - rcj[0]) + (rci[1] - rcj[1])) * rdj[0];
      const float x1 = rp[1] * __builtin_amdgcn_exp2f((rci[0] - rcj[2]) + (rci[1] - rcj[3])) * rdj[1];
      uint32_t p[3];
      cut3(x0, pcol + 1 < prow ? x1 : 0.f, p);
#pragma unroll
      for (int m = 0; m < 3; ++m) *reinterpret_cast<uint32_t*>(lds + b * IMG + M_AT + m * MAT + pair_at(prow, pcol)) = p[m];
    }
  };

  // state: lane (col, g) holds column nc, key channels 32 s + 8 g .. + 7 in blocks 2 s, 2 s + 1
  float* st = a.state + (((int64_t)seq.slot * a.H + h) * a.dv + nc) * DK + 8 * g;
  f32x4 S[NB];
  const auto load = [&](const float* from) {
#pragma unroll
    for (int b = 0; b < NB; ++b) S[b] = *reinterpret_cast<const f32x4*>(from + 32 * (b >> 1) + 4 * (b & 1));
  };
  const auto store = [&](float* to) {
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<f32x4*>(to + 32 * (b >> 1) + 4 * (b & 1)) = S[b];
  };
  const auto finite = [&] {   // of the whole wave's S
    float broken = 0.f;       // NaN if a value of S is not finite
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int e = 0; e < 4; ++e) broken += S[nb][e] * 0.f;
    return __ballot(broken != 0.f) == 0;
  };
  const auto zero = [&] {
#pragma unroll
    for (int b = 0; b < NB; ++b) S[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  const int64_t o_step = (int64_t)RC * 2 * a.out_stride;
  const int64_t mine = (int64_t)nc * DK + 8 * g, copy = (int64_t)a.dv * DK;   // places in a segment's floats
  const float Dh = DELTA ? 0.f : a.D[h];
  // outputs: lane (col, g) holds rows col and 16 + col, columns n0 + 4 g .. + 3
  char* op = reinterpret_cast<char*>(a.out + (int64_t)r0 * a.out_stride + (int64_t)h * a.dv + c0);
  const uint32_t ol = 2 * (16 * wave + 4 * g);
  const uint32_t oo[2] = {2 * (uint32_t)col * (uint32_t)a.out_stride, 2 * (uint32_t)(16 + col) * (uint32_t)a.out_stride};

  // the sequence row by row, as the row-by-row kernels do it (each lane its 8 key channels of every 32)
  const auto walk = [&](int from, int to, bool write) {
    for (int64_t row = from; row < to; ++row) {
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
      if (write && live && g == 0) a.out[row * a.out_stride + (int64_t)h * a.dv + nc] = (bf16)(DELTA ? decay * sq + add * kq : sq + Dh * x);
    }
  };

  // what the sequence starts from
  const auto origin = [&] {
    if (SEG == 2 && !(last && j == 0)) load(sg - j * sg_step + copy + mine);   // (its last segment may have written `state` by now)
    else if (seq.fresh) zero();
    else load(st);
  };
  // what the rows r0 and up start from
  const auto start = [&] {
    if (SEG == 2 && j > 0) {
      const float* f = sg - j * sg_step;
      load(f + mine);
#pragma unroll 1
      for (int i = 1; i < j; ++i) {
        f += sg_step;
        if constexpr (DELTA) {   // S = M S + S_i, M through LDS (16-byte pieces swizzled by the rows that a product takes together)
          if (i > 1) __syncthreads();
          constexpr int PR = DK / 4;   // pieces of a row
#pragma unroll
          for (int x = 0; x < DK * DK / 256 / NW; ++x) {
            const int e = 64 * (wave + NW * x) + lane, row = e / PR;
            buffer_to_lds(f + copy, 4 * DK * DK, 4 * row * DK + 16 * ((e % PR) ^ ((row & 3) | ((row >> 3) & 3) << 2)), 0, lds0 + 1024 * (wave + NW * x));
          }
          f32x4 n[NB];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) n[nb] = *reinterpret_cast<const f32x4*>(f + mine + 32 * (nb >> 1) + 4 * (nb & 1));
          bf16x8 part[NS][3];
#pragma unroll
          for (int t = 0; t < NS; ++t) split3(S[2 * t], S[2 * t + 1], part[t]);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          __syncthreads();
          const float* m = reinterpret_cast<const float*>(lds) + (8 * (col >> 2) + (col & 3)) * DK;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const float* r = m + (32 * (nb >> 1) + 4 * (nb & 1)) * DK;
            bf16x8 x[NS][3];
#pragma unroll
            for (int t = 0; t < NS; ++t)
              split3(*reinterpret_cast<const f32x4*>(r + 4 * ((8 * t + 2 * g) ^ col)), *reinterpret_cast<const f32x4*>(r + 4 * ((8 * t + 2 * g + 1) ^ col)), x[t]);
            f32x4 ms = {0.f, 0.f, 0.f, 0.f};   // the smallest terms first
#pragma unroll
            for (int sum = 2; sum >= 0; --sum)
#pragma unroll
              for (int t = 0; t < NS; ++t)
#pragma unroll
                for (int y = 0; y <= sum; ++y) ms = mma_bf16(x[t][y], part[t][sum - y], ms);
            S[nb] = ms + n[nb];
          }
        } else {
          const float d = f[copy];
#pragma unroll
          for (int b = 0; b < NB; ++b) S[b] = S[b] * d + *reinterpret_cast<const f32x4*>(f + mine + 32 * (b >> 1) + 4 * (b & 1));
        }
      }
      if (DELTA && j > 1) __syncthreads();
      if (live && !finite()) {   // row by row, as the sequence in one piece has it
        origin();
        walk(q0, r0, false);
      }
    } else if (SEG == 1 && j > 0) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[b][e] = ident && 32 * (b >> 1) + 8 * g + 4 * (b & 1) + e == nc ? 1.f : 0.f;
    } else {
      origin();
      if (SEG == 1 && live) store(sg + copy + mine);
    }
  };
  start();

  if (!few) {
    if constexpr (MW == 0) {
      offsets(min(RC, r1 - r0));
      move(RC, true, 0);
    }
    ahead(0);
    advance(chunks > 1);
    if constexpr (!DELTA && SEG != 1) {   // the rest of P, of which every thread has as much (a row and a column from the other end): zero
#pragma unroll
      for (int m = 0; m < 6; ++m) *reinterpret_cast<uint32_t*>(lds + m / 3 * IMG + M_AT + m % 3 * MAT + pair_at(31 - prow, 30 - pcol)) = 0;
    }
    put(0);
    if constexpr (MW == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  float decay = 1.f;   // of the chunks so far (SEG 1, Mamba-2)
  // One chunk.  With one or two waves a SIMD nothing else covers an LDS read: each is issued a stage before its use, and the
  // scheduling barriers keep the compiler from sinking it there.
  const auto step = [&](int c, int b) {
    const char* L = lds + b * IMG;
    const bf16 *K = reinterpret_cast<const bf16*>(L), *Q = reinterpret_cast<const bf16*>(L + ROWS), *X = reinterpret_cast<const bf16*>(L + X_AT);
    const float* V = reinterpret_cast<const float*>(L + V_AT);
    const auto vec = [&](int i, int rb) { return *reinterpret_cast<const f32x4*>(V + i * RC + 16 * rb + 4 * g); };
    const auto mat = [&](int m, int rb) { return *reinterpret_cast<const bf16x8*>(L + M_AT + m * MAT + mat_img(16 * rb + col, g)); };
    const auto rows = [&](const bf16* R, int rb, int t) { return ld8(R + img<DK>(16 * rb + col, 4 * t + g) * 8); };
    // ---- first operands ----
    bf16x4 x[2], y[2];
    f32x4 va[2], vb[2], vd[2];
    bf16x8 kf[2][NS], qf[2][NS];
    const float gc = V[(DELTA ? 4 : 6) * RC];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
        if constexpr (DELTA) kf[rb][t] = rows(K, rb, t);
        else if constexpr (SEG != 1) qf[rb][t] = rows(Q, rb, t);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      x[rb] = tr4(X, 8 * val_img(16 * rb + 4 * g + (col >> 2), 2 * wave + ((col >> 1) & 1)) + 4 * (col & 1));
      if constexpr (DELTA) {
        va[rb] = vec(0, rb);
        vb[rb] = vec(1, rb);
      }
    }
    if constexpr (MW == 0) move(r1 - r0 - (c + 1) * RC, c + 1 < chunks, b ^ 1);   // (that buffer was read last before the previous barrier)
    ahead(min(c + 1, chunks - 1));
    advance(c + 2 < chunks);
    if constexpr (DELTA && SEG != 1) {
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) qf[rb][t] = rows(Q, rb, t);
    }
    __builtin_amdgcn_sched_barrier(0x0f);
    // ---- S in three parts; k S ----
    f32x4 ks[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    bf16x8 part[NS][3];
#pragma unroll
    for (int t = 0; t < NS; ++t) {   // (S is scaled first: what a rounding leaves is computed in the place of its value)
      const f32x4 s0 = S[2 * t], s1 = S[2 * t + 1];
      S[2 * t] *= gc;
      S[2 * t + 1] *= gc;
      if constexpr (DELTA || SEG != 1) split3(s0, s1, part[t]);
      if constexpr (DELTA) {
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) ks[rb] = mma_bf16(kf[rb][t], part[t][p], ks[rb]);
      }
    }
    __builtin_amdgcn_sched_barrier(0x0f);
    // ---- q S (transposed); R (DELTA) / U (Mamba-2) ----
    bf16x8 tm[2][3], pm[2][3];
    float vo[2], vp[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        if constexpr (DELTA || SEG != 1) tm[rb][p] = mat(p, rb);
      vo[rb] = V[(DELTA ? 2 : 3) * RC + 16 * rb + col];
      if constexpr (!DELTA && SEG != 1) vp[rb] = V[5 * RC + 16 * rb + col];
      vd[rb] = vec(DELTA ? 3 : 4, rb);
    }
    __builtin_amdgcn_sched_barrier(0x0f);
    if constexpr (SEG != 1) {
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) o[rb] = mma_bf16(part[t][p], qf[rb][t], o[rb]);
    }
    f32x4 r[2], u[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[rb][e] = DELTA ? va[rb][e] * (float)x[rb][e] - vb[rb][e] * ks[rb][e] : (float)x[rb][e];
      }
    bf16x8 rs[3];
    if constexpr (DELTA) split3(r[0], r[1], rs);
    __builtin_amdgcn_sched_barrier(0x0f);
    // ---- U = T R, o += (P T) R (Mamba-2: o += P dt x) ----
    bf16x8 ka[NB];
    {
      const int qr = 4 * g + (col >> 2), p4 = col & 3;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int ch = 4 * (nb >> 1) + p4, half = 4 * (nb & 1);
        const bf16x4 lo = tr4(K, img<DK>(qr, ch) * 8 + half), hi = tr4(K, img<DK>(16 + qr, ch) * 8 + half);
        ka[nb] = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
#pragma unroll
    for (int rb = 0; SEG != 1 && rb < 2; ++rb) {
      if constexpr (DELTA) {
#pragma unroll
        for (int p = 0; p < 3; ++p) pm[rb][p] = mat(3 + p, rb);
      } else {
        y[rb] = *reinterpret_cast<const bf16x4*>(X + 8 * val_img(16 * rb + col, 2 * wave + (g >> 1)) + 4 * (g & 1));
      }
    }
    __builtin_amdgcn_sched_barrier(0x0f);
    if constexpr (DELTA) mma_parts(tm, rs, u);
    if constexpr (SEG != 1) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) o[rb] *= vo[rb];
      if constexpr (DELTA) {
        mma_parts<true>(pm, rs, o);
      } else {   // the values as they are
        const bf16x8 xv = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) o[rb] = mma_bf16(xv, tm[rb][p], o[rb]);
      }
    }
    // ---- S = g_C S + k^T U ----
    bf16x8 us[3];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) u[rb] = (DELTA ? u[rb] : r[rb]) * vd[rb];
    split3(u[0], u[1], us);
    constexpr bool BESIDE = SEG == 0 && (DELTA || MW == 0);   // the outputs' vector instructions beside S's products
    if constexpr (BESIDE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) S[nb] = mma_bf16(ka[nb], us[p], S[nb]);
    if constexpr (SEG == 1) {
      if constexpr (!DELTA) decay *= gc;
      if constexpr (MW == 0) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next chunk has landed
      }
      __syncthreads();
      return;
    }
    // ---- the outputs ----
    if constexpr (!DELTA) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int t = 0; t < 4; ++t) o[rb][t] += (Dh + vp[rb]) * (float)y[rb][t];
    }
    put(b ^ 1);
    if constexpr (BESIDE) {   // (a delta rule's chunk alone on its CU 1.48 -> 1.42 us, selective scan of 512 workgroups 75 -> 74; segments 0.5%, a selective scan with waves that move 4% slower so)
#pragma unroll
      for (int i = 0; i < 3 * NB; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MW == 0) {
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next chunk has landed (before the stores below, which nobody waits for)
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const bool in = live && 16 * rb + col < r1 - r0 - c * RC;
      const bf16x4 v = {(bf16)o[rb][0], (bf16)o[rb][1], (bf16)o[rb][2], (bf16)o[rb][3]};
      if constexpr (VEC) {   // (rows past the end: an offset past the descriptor's, so not stored)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), __builtin_amdgcn_make_buffer_rsrc(op, 0, 0x7fffffff, 0x00020000),
                                              in ? oo[rb] + ol : 0x80000000u, 0, 0);
      } else if (in) {
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<bf16*>(op + oo[rb] + ol + 2 * e) = v[e];
      }
    }
    op += o_step;
    __syncthreads();
  };
  for (int c = 0; !few && c < chunks; c += 2) {
    step(c, 0);
    if (c + 1 < chunks) step(c + 1, 1);
  }
  if constexpr (SEG == 1) {
    if (ident) {   // M by rows: lane (col, g) holds column nc
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) sg[copy + (32 * (b >> 1) + 8 * g + 4 * (b & 1) + e) * DK + nc] = S[b][e];
    } else if (live) {
      store(sg + mine);
      if (!DELTA && j > 0 && tid == 0 && blockIdx.y == 0) sg[copy] = decay;
    }
    return;
  }
  if (live && (few || !finite())) {
    if (!few) {
      origin();
      walk(q0, r0, false);
    }
    walk(r0, r1, true);
  }
  if (live && last) store(st);
}

bool aligned16(const void* p, int64_t elems) { return ((uintptr_t)p | (uintptr_t)(elems * 2)) % 16 == 0; }

template <bool DELTA>
int launch_rule(RuleArgs a, int T, int dk, hipStream_t stream) {
  const bool vec = aligned16(a.v, a.v_stride) && ((uintptr_t)a.out | (uintptr_t)(2 * a.out_stride)) % 8 == 0;   // (dv is a multiple of 16)
  if (!vec) a.seg = 0;
  char* end = a.ws + (int64_t)(T / RC + a.S) * ws_bytes<DELTA>(a.H, a.Hk);
  a.turn = a.S > 1 && a.S <= TURNS && !a.seg ? reinterpret_cast<int4*>(end) : nullptr;
  a.segs = reinterpret_cast<float*>(end);
  const int cols = (a.dv + 63) / 64, ids = a.seg ? T / (RC * a.seg) + a.S : a.S;
  if (ids > 65535) return -3;
  const bool alone = (int64_t)a.H * cols * ids <= 256;   // one workgroup a CU at most: waves that move (chunk_rule_kernel)
  const dim3 gram(T / RC + a.S, DELTA ? (a.H + 3) / 4 : a.Hk), rule(a.H, cols, ids), own(a.H, cols + (DELTA ? dk / 64 : 0), ids);
#define CHUNKS(DK)                                                                                                      \
  {                                                                                                                     \
    if constexpr (DELTA) chunk_gram_kernel<DK><<<gram, 256, 0, stream>>>(a);                                            \
    else ssm_gram_kernel<DK><<<gram, 256, 0, stream>>>(a);                                                              \
    if (vec && a.seg) {                                                                                                 \
      chunk_rule_kernel<DK, DELTA, 4, true, 1, 4><<<own, 64 * 8, 0, stream>>>(a);                                       \
      if (alone) chunk_rule_kernel<DK, DELTA, 4, true, 2, 2><<<rule, 64 * 6, 0, stream>>>(a);                           \
      else chunk_rule_kernel<DK, DELTA, 4, true, 2, 0><<<rule, 256, 0, stream>>>(a);                                    \
    } else if (!vec) chunk_rule_kernel<DK, DELTA, 4, false, 0, 0><<<rule, 256, 0, stream>>>(a);                         \
    else if (alone) chunk_rule_kernel<DK, DELTA, 4, true, 0, 2><<<rule, 64 * 6, 0, stream>>>(a);                        \
    else chunk_rule_kernel<DK, DELTA, 4, true, 0, 0><<<rule, 256, 0, stream>>>(a);                                      \
  }
  if (dk == 128) CHUNKS(128)
  else CHUNKS(64)
#undef CHUNKS
  OME_CHECK_LAUNCH();
  return 0;
}

// (row strides below 2^24 elements: a chunk's byte offsets stay in 32 bits)
bool rule_shape(int S, int H, int Hk, int dk, int dv, int64_t s0, int64_t s1, int64_t s2) {
  return s0 >= 0 && s1 >= 0 && s2 >= 0 && s0 < 1 << 24 && s1 < 1 << 24 && s2 < 1 << 24 && S > 0 && S <= 65535 && H > 0 && Hk > 0 && H % Hk == 0 && (dk == 64 || dk == 128) && dv > 0 && dv % 16 == 0 &&
         (dv + 63) / 64 <= 65535 && H <= 65535;
}

}  // namespace

// fp32 words of workspace of one chunk of H heads (Mamba-2: in G groups); T rows of S sequences have up to T / 32 + S
OME_API int ome_chunk_rule_floats(int H, int G, int delta) {
  return (int)((delta ? ws_bytes<true>(H, G) : ws_bytes<false>(H, G)) / 4);
}

// ... and of a head of a segment, of which there are up to T / (32 seg) + S; they come behind the chunks' (without segments: 256 words, the order)
OME_API int ome_chunk_rule_seg_floats(int dk, int dv) { return (int)seg_floats(dv, dk); }

// Gated delta rule over all rows of every sequence, in segments of `seg` chunks (0: in one piece); operands as ome_gdn_scan.  -3: a shape, stride or
// alignment that the chunked kernels do not take (nothing is launched).
OME_API int ome_gdn_chunks(const void* q, const void* k, const void* v, int64_t qkv_stride, const void* a, const void* b,
                           int64_t ab_stride, const float* A_log, const float* dt_bias, float* state, void* out,
                           int64_t out_stride, const int* cu, const int* slot, const int* reset, int S, int T, int Hv, int Hk,
                           int dk, int dv, int seg, float* ws, hipStream_t stream) {
  if (T <= 0 || seg < 0 || !ws || !rule_shape(S, Hv, Hk, dk, dv, qkv_stride, qkv_stride, out_stride) || !aligned16(q, qkv_stride) || !aligned16(k, qkv_stride) ||
      (uintptr_t)state % 16 || (uintptr_t)ws % 16)
    return -3;
  const RuleArgs r{(const bf16*)q, (const bf16*)k, (const bf16*)v, qkv_stride, qkv_stride, (const bf16*)a, (const bf16*)b,
                   ab_stride, A_log, nullptr, dt_bias, 0.f, (char*)ws, state, (bf16*)out, out_stride, cu, slot, reset, S, Hv, Hk, dv, seg, nullptr, nullptr};
  return launch_rule<true>(r, T, dk, stream);
}

// Mamba-2's selective scan over all rows of every sequence; operands as ome_ssm_scan.
OME_API int ome_ssm_chunks(const void* x, int64_t x_stride, const void* dt, int64_t dt_stride, const void* B, const void* Cm,
                           int64_t bc_stride, const float* A, const float* D, const float* dt_bias, float dt_min, float* state,
                           void* y, int64_t y_stride, const int* cu, const int* slot, const int* reset, int S, int T, int H,
                           int P, int N, int G, int seg, float* ws, hipStream_t stream) {
  if (T <= 0 || seg < 0 || !ws || !rule_shape(S, H, G, N, P, bc_stride, x_stride, y_stride) || !aligned16(B, bc_stride) || !aligned16(Cm, bc_stride) ||
      (uintptr_t)state % 16 || (uintptr_t)ws % 16)
    return -3;
  const RuleArgs r{(const bf16*)Cm, (const bf16*)B, (const bf16*)x, bc_stride, x_stride, (const bf16*)dt, nullptr,
                   dt_stride, A, D, dt_bias, dt_min, (char*)ws, state, (bf16*)y, y_stride, cu, slot, reset, S, H, G, P, seg, nullptr, nullptr};
  return launch_rule<false>(r, T, N, stream);
}
