// Batch-1..8 decode GEMV for gfx950: out[M, N] = X[M, K] . W[N, K]^T (+ bias), M <= 8
// (decode-skinny shapes at the low end of the BenchmarkJob concurrency sweep).
//
// At one to four rows a projection has no operand reuse worth an MFMA tile: it is a pure
// HBM stream of the weight.  Each wave owns R consecutive weight rows and walks K with 16-byte
// loads (lane l covers k = 8 l + 512 i), the R row loads of several K steps in flight at once
// (unrolled; no LDS, no barriers, ~30 VGPRs so many waves per SIMD hide the HBM latency).  The
// activation rows (<= 8 x K bf16, read by every wave) are served by L1 / L2.  Each wave reduces
// its M x R fp32 partial dot products across the 64 lanes with xor shuffles and stores them.
#include "common.h"

namespace {

// 8-element bf16 dot product on four v_dot2c_f32_bf16 (fp32 accumulate, no unpacking)
__device__ __forceinline__ float dot8(bf16x8 a, bf16x8 b, float acc) {
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(a, a, 0, 1), __builtin_shufflevector(b, b, 0, 1), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(a, a, 2, 3), __builtin_shufflevector(b, b, 2, 3), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(a, a, 4, 5), __builtin_shufflevector(b, b, 4, 5), acc, false);
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(a, a, 6, 7), __builtin_shufflevector(b, b, 6, 7), acc, false);
}

// SwiGLU operand on the fly: X holds [gate | up] (2K wide); the dot product sees
// bf16(silu(g) * u), bit-identical to act_and_mul followed by the plain GEMV.
__device__ __forceinline__ bf16x8 silu_mul8(bf16x8 g, bf16x8 u) {
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float gf = (float)g[j];
    o[j] = (bf16)(gf / (1.f + __expf(-gf)) * (float)u[j]);
  }
  return o;
}

template <bool ACT>
__device__ __forceinline__ bf16x8 ldx8(const bf16* p, int K) {
  if constexpr (ACT) return silu_mul8(ld8(p), ld8(p + K));
  else return ld8(p);
}

// What follows a projection element by element is done by the wave that holds its sums.  At one to four rows a launch of
// its own costs near 4.6 us whatever it does, against 41 us (gate_up) or 12 us (QKV) of weight stream (Llama-3-8B):
//   SWIGLU: W is gate / up interleaved in 16-row blocks; a wave takes R / 2 gate rows and their up rows.
//   QKV:    a wave takes R / 2 dims d of a head and their partners d + D / 2, rotates them and writes q or the cache.
// Both round the projection to bf16 first, as its own store did: the results are the same bits.
//   ADD:    out += the projection, the residual stream's sum ahead of a norm that is folded into the next product (gemm_rows.hip).
// A decode step of one request (Llama-3-8B, 700 tokens of context): 3.69 -> 3.57 ms with the first two.
enum { PLAIN = 0, SWIGLU = 1, QKV = 2, ADD = 3 };
struct GemvQkv {
  const int *positions, *slots;
  const float* cos_sin;
  bf16* q;
  void *k, *v;
  int Hq, Hkv, D;   // pages of 16 tokens: k [page][head][16][D], v [page][head][D][16]
  float k_inv, v_inv;
};

// weight row r of the R rows of a wave that begins at row (PLAIN, ADD) or output pair n0 / 2
template <int R, int EPI>
__device__ __forceinline__ int weight_row(int n0, int r, int N, int D) {
  if constexpr (EPI == PLAIN || EPI == ADD) return min(n0 + r, N - 1);   // clamp: rows past N are computed, not stored
  const int p = n0 / 2 + r % (R / 2), up = r / (R / 2);
  if constexpr (EPI == SWIGLU) return 32 * (p >> 4) + (p & 15) + 16 * up;
  const int half = D >> 1;
  return p / half * D + p % half + up * half;
}

// Weights are read once, so they come with the non-temporal policy and leave the rows in the caches: QKV of one row 14.0 -> 13.7 us, 4096 x 4096 9.5 ->
// 9.4, a whole step of one request 3342 -> 3231 (two runs of one side differ by 2%).
__device__ __forceinline__ bf16x8 ld8_once(const bf16* p) { return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p)); }

template <int M, int R, int U, bool ACT = false, int EPI = PLAIN, int F = KV_BF16>   // U: K steps in flight (fewer for more rows: VGPR budget)
__global__ __launch_bounds__(256) void gemv_kernel(const bf16* __restrict__ X, int64_t ldx, const bf16* __restrict__ W,
                                                   const bf16* __restrict__ bias, bf16* __restrict__ out, int64_t ldo,
                                                   int N, int K, GemvQkv e) {
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
  if (n0 >= N) return;
  const bf16* wr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) wr[r] = W + (int64_t)weight_row<R, EPI>(n0, r, N, e.D) * K;
  // QKV: this lane's element (row em, weight row er) and its rotation, read ahead of the weight stream
  const int em = min(lane / R, M - 1), er = lane % R;
  int head = 0, dim = 0, slot = 0;
  float c = 1.f, sn = 0.f;
  if constexpr (EPI == QKV) {
    const int n = weight_row<R, EPI>(n0, er, N, e.D), half = e.D >> 1;
    head = n / e.D;
    dim = n % e.D;
    slot = e.slots[em];
    if (head < e.Hq + e.Hkv) {
      const float* cs = e.cos_sin + (int64_t)e.positions[em] * e.D + (dim >= half ? dim - half : dim);
      c = cs[0];
      sn = cs[half];
    }
  }
  float before = 0.f;   // ADD: of this lane's element
  if constexpr (EPI == ADD) before = (float)out[(int64_t)em * ldo + min(n0 + er, N - 1)];
  float acc[M][R];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.f;

  int k = lane * 8;
  // main body: U K steps (U x R 16-B weight loads per lane) in flight
  for (; k + (U - 1) * 512 < K; k += U * 512) {
    bf16x8 w[U][R], x[U][M];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) w[u][r] = ld8_once(wr[r] + k + 512 * u);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < M; ++m) x[u][m] = ldx8<ACT>(X + m * ldx + k + 512 * u, K);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[m][r] = dot8(x[u][m], w[u][r], acc[m][r]);
  }
  for (; k < K; k += 512) {
    bf16x8 w[R], x[M];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = ld8_once(wr[r] + k);
#pragma unroll
    for (int m = 0; m < M; ++m) x[m] = ldx8<ACT>(X + m * ldx + k, K);
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[m][r] = dot8(x[m], w[r], acc[m][r]);
  }
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = wave_sum(acc[m][r]);
  // lane (m * R + r) stores element (m, n0 + r)
  if constexpr (EPI == PLAIN) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (lane == m * R + r && n0 + r < N)
          out[(int64_t)m * ldo + n0 + r] = (bf16)(acc[m][r] + (bias ? (float)bias[n0 + r] : 0.f));
  } else if constexpr (EPI == ADD) {
    float x = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) x = lane == m * R + r ? acc[m][r] : x;
    if (lane < M * R && n0 + er < N) out[(int64_t)em * ldo + n0 + er] = (bf16)(before + (float)(bf16)x);
  } else if constexpr (EPI == SWIGLU) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R / 2; ++r) {
        const float gt = (float)(bf16)acc[m][r], up = (float)(bf16)acc[m][r + R / 2];
        if (lane == m * R + r) out[(int64_t)m * ldo + n0 / 2 + r] = (bf16)(gt / (1.f + __expf(-gt)) * up);
      }
  } else {
    float x = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) x = lane == m * R + r ? acc[m][r] : x;
    x = (float)(bf16)(x + (bias ? (float)bias[head * e.D + dim] : 0.f));
    const float y = __shfl_xor(x, R / 2);   // the rotation's other element
    if (lane < M * R) {
      const int64_t page = slot >> 4, off = slot & 15;
      typedef typename KVStore<F>::T T;
      if (head < e.Hq + e.Hkv) x = dim < (e.D >> 1) ? x * c - y * sn : x * c + y * sn;
      if (head < e.Hq) {
        e.q[((int64_t)em * e.Hq + head) * e.D + dim] = (bf16)x;
      } else if (slot >= 0) {
        const int kh = head - e.Hq;
        if (kh < e.Hkv)
          kv_st1<F>((T*)e.k + ((page * e.Hkv + kh) * 16 + off) * e.D + dim, F == KV_BF16 ? x : (float)(bf16)x * e.k_inv);
        else
          kv_st1<F>((T*)e.v + ((page * e.Hkv + kh - e.Hkv) * e.D + dim) * 16 + off, F == KV_BF16 ? x : x * e.v_inv);
      }
    }
  }
}

}  // namespace

// X [M, K] (row stride ldx, 16-byte aligned rows), W [N, K] contiguous, out [M, N] (row stride ldo);
// 1 <= M <= 8, K % 8 == 0.  act = 1: X is the fused gate/up projection [M, 2K] and the operand is
// SiLU(gate) * up (the down projection with the SwiGLU folded into its operand load).
template <bool ACT, int EPI = PLAIN, int F = KV_BF16>
static int gemv_launch(const void* X, int64_t ldx, const void* W, const void* bias, void* out, int64_t ldo, int M,
                       int N, int K, hipStream_t stream, const GemvQkv& e = GemvQkv{}) {
  // narrow weights: 2 rows per wave (twice the waves to spread over 256 CUs); long rows (K >= 8192,
  // the down projection) with <= 2 activation rows: 8 K steps in flight per wave
  const bool narrow = N <= 4096, deep = K >= 8192 && M <= 2;
#define GV_L(MV, RV, UV)                                                                                    \
  gemv_kernel<MV, RV, UV, ACT, EPI, F><<<dim3((N + 4 * RV - 1) / (4 * RV)), 256, 0, stream>>>(                     \
      (const bf16*)X, ldx, (const bf16*)W, (const bf16*)bias, (bf16*)out, ldo, N, K, e)
#define GV(MV)                                                                              \
  if (MV <= 2 && deep) { if (narrow) GV_L(MV, 2, 8); else GV_L(MV, 4, 8); }                \
  else if (narrow) GV_L(MV, 2, (MV <= 4 ? 4 : 2));                                          \
  else GV_L(MV, 4, (MV <= 4 ? 4 : 2))
  switch (M) {
    case 1: GV(1); break;
    case 2: GV(2); break;
    case 3: GV(3); break;
    case 4: GV(4); break;
    case 5: GV(5); break;
    case 6: GV(6); break;
    case 7: GV(7); break;
    default: GV(8); break;
  }
#undef GV_L
#undef GV
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_gemv(const void* X, int64_t ldx, const void* W, const void* bias, void* out, int64_t ldo, int M, int N,
                     int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 8 || K % 8 || ldx % 8 || K <= 0) return -2;
  return gemv_launch<false>(X, ldx, W, bias, out, ldo, M, N, K, stream);
}

// out [M, N] += X . W^T, the product and the sum each rounded to bf16
OME_API int ome_gemv_add(const void* X, int64_t ldx, const void* W, void* out, int64_t ldo, int M, int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 8 || K % 8 || ldx % 8 || K <= 0) return -2;
  return gemv_launch<false, ADD>(X, ldx, W, nullptr, out, ldo, M, N, K, stream);
}

OME_API int ome_gemv_act(const void* X, int64_t ldx, const void* W, const void* bias, void* out, int64_t ldo, int M,
                         int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 8 || K % 8 || ldx % 8 || K <= 0 || ldx < 2 * (int64_t)K) return -2;
  return gemv_launch<true>(X, ldx, W, bias, out, ldo, M, N, K, stream);
}


// out [M, I] = SiLU(X . Wg^T) * (X . Wu^T); W [2 I, K]: gate and up rows alternate in blocks of 16 (I % 16 == 0)
OME_API int ome_gemv_swiglu(const void* X, int64_t ldx, const void* W, void* out, int64_t ldo, int M, int I, int K,
                            hipStream_t stream) {
  if (M <= 0 || I <= 0) return 0;
  if (M > 8 || I % 16 || K % 8 || ldx % 8 || K <= 0) return -2;
  return gemv_launch<false, SWIGLU>(X, ldx, W, nullptr, out, ldo, M, 2 * I, K, stream);
}

// X . W^T (+ bias), W [(Hq + 2 Hkv) D, K]; q [M, Hq, D] rotated, k rotated and v into the paged cache at slots[m]
// (slot < 0: neither).  The whole head rotates (cos_sin rows of D floats); kv_fmt, scales: as ome_rope_qkv_cache.
OME_API int ome_gemv_qkv(const void* X, int64_t ldx, const void* W, const void* bias, const int* positions,
                         const float* cos_sin, void* q, void* k_cache, void* v_cache, const int* slots, int M, int Hq,
                         int Hkv, int D, int P, int K, int kv_fmt, float k_scale, float v_scale, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 8 || K % 8 || ldx % 8 || K <= 0 || Hq <= 0 || Hkv <= 0) return -2;
  if ((D != 128 && D != 64 && D != 256) || P != 16) return -4;
  const GemvQkv e{positions, slots, cos_sin, (bf16*)q, k_cache, v_cache, Hq, Hkv, D, 1.f / k_scale, 1.f / v_scale};
  const int N = (Hq + 2 * Hkv) * D;
  if (kv_fmt == KV_BF16) return gemv_launch<false, QKV, KV_BF16>(X, ldx, W, bias, nullptr, 0, M, N, K, stream, e);
  if (kv_fmt == KV_E4M3) return gemv_launch<false, QKV, KV_E4M3>(X, ldx, W, bias, nullptr, 0, M, N, K, stream, e);
  if (kv_fmt == KV_E5M2) return gemv_launch<false, QKV, KV_E5M2>(X, ldx, W, bias, nullptr, 0, M, N, K, stream, e);
  return -5;
}
