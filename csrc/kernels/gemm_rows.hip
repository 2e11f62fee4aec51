// Projections of up to 256 rows (decode steps, short prompts), bf16:  X[M][K] . W[N][K]^T  (= F.linear(x, w)).
//
// What bounds it: the weights, which a launch of 200 workgroups and more reads at 5.5 to 6 TB/s however little of them each has in
// flight, and the rows, which every workgroup reads again from L2.  The two add up: 28672 x 4096 alone takes 39 us, 256 rows
// alone 17 (64 bytes a clock and CU), both 55, whatever the depth and whichever waves move them.  Hence
//   * a workgroup takes ALL rows of 128 columns: no weight is fetched twice, and a row's bytes serve 128 columns;
//   * K is cut into as many pieces as fill the chip (`splits`).  The next kernel adds their fp32 sums as it reads them
//     (ome_add_rmsnorm_parts): no second step at the tail of this one, where most CUs would have left;
//   * weights come with the non-temporal policy, so the rows stay in L2 (28672 x 4096, 256 rows: 66 -> 60 us), and workgroups start
//     at different places in K: in step, all would read the same 128 bytes of rows a power of two apart, which are few
//     of the memory's channels (weights alone: 48 -> 39 us);
//   * rows past M are outside their descriptor: they arrive as zeros and are never fetched.
// us, weights cold, stream-K or library -> this (without the addition):   rows 20          64          128         200         256
//   28672 x 4096, SiLU * up in the epilogue (no pieces)           48 -> 37    49 -> 38    52 -> 46    64 -> 57    66 -> 60
//   4096 x 14336 (8 pieces)                                       28 -> 20    40 -> 22    37 -> 27    44 -> 34    49 -> 37
//   4096 x 4096 (8 pieces)                                        20 -> 8.5   20 -> 9.5   19 -> 12    22 -> 17    22 -> 21
#include "common.h"

namespace {

typedef __attribute__((address_space(3))) void lds_void_t;
enum { GR_BF16 = 0, GR_SILU = 2, GR_PART = 3 };

constexpr int BN = 128;

__device__ __forceinline__ int gr_swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// (non-template wrappers: the builtin exists for the device target only)
__device__ __forceinline__ void gr_to_lds(__amdgpu_buffer_rsrc_t rs, char* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void gr_to_lds_nt(__amdgpu_buffer_rsrc_t rs, char* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)lds, 16, voff, soff, 0, 2);
}

// WM x WN waves; a wave owns 16 FR rows and BN / WN columns.  A step of 64 k has two phases of matrix instructions; the barrier that
// publishes the next tile stands between them.  Tile t's weights are asked for in the second phase of step t - NST, its rows in the
// first one of step t - NST + 1.
// NORM: X holds one or two rows of the residual stream, and out is the product of their RMSNorm (weights `ln`).  Every workgroup forms the norm itself,
// in LDS, while its first weights are on their way: no rows move with the weights.  One row, 28672 x 4096: 4.6 + 38.1 us -> 39.1 (scaled between LDS
// and the products instead 39.4, its loads ahead of the weights' 39.3, two more stages 39.6).
// The squares are added in the order of fused_add_rmsnorm_kernel of 8 waves, which these rows take elsewhere: the norm is the same bits.
constexpr int LN_ROWS = 2, LN_K = 8192, LN_WAVES = 8;   // rows and K at most
template <int WM, int WN, int FR, int NST, int EPI, bool NORM = false>
__global__ __launch_bounds__(64 * WM * WN, WM * WN / 4) void gemm_rows_kernel(
    const bf16* __restrict__ X, int64_t ldx, const bf16* __restrict__ W, int64_t ldw, const bf16* __restrict__ bias,
    bf16* __restrict__ out, int64_t ldo, int M, int N, int steps, int splits, float* __restrict__ part, const bf16* __restrict__ ln, float eps) {
  constexpr int NW = WM * WN, BM = 16 * FR * WM, NI = BN / 16 / WN;
  constexpr int PW = BN / 8 / NW, PX = NORM ? 0 : BM / 8 / NW, LPT = PW + PX;   // moves of 1 KB (8 rows) per wave and step
  constexpr int BUF = (BN + (NORM ? 0 : BM)) * 128, XAT = BN * 128;
  static_assert(PW * NW * 8 == BN && (NORM || (PX * NW * 8 == BM && PX > 0)) && NI > 0 && (EPI != GR_SILU || NI % 2 == 0), "tile");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, fr = lane & 15, fc = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int sp = blockIdx.x % splits, tile = blockIdx.x / splits, n0 = tile * BN;
  const int t0 = (int)((int64_t)steps * sp / splits), n = (int)((int64_t)steps * (sp + 1) / splits) - t0;

  uint32_t wo[PW], xo[NORM ? 1 : PX];
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const int r = (wave * PW + j) * 8 + (lane >> 3);
    wo[j] = 2 * (uint32_t)(r * ldw) + 16 * gr_swz(r, lane & 7);
  }
#pragma unroll
  for (int j = 0; j < PX; ++j) {
    const int r = (wave * PX + j) * 8 + (lane >> 3);
    xo[j] = 2 * (uint32_t)(r * ldx) + 16 * gr_swz(r, lane & 7);
  }
  const bf16* Wt = W + (int64_t)n0 * ldw;
  const int xbytes = (int)(2 * ((M - 1) * ldx + 64 * (int64_t)steps));
  // step s of the workgroup is K tile t0 + (s + tile) mod n; steps past its n read nothing (an empty descriptor; counted all the same)
  int sw = 0, kw = tile % n, sx = 0, kx = kw;
  const auto load_w = [&](int b) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)Wt, (short)0, sw < n ? 0x7fffffff : 0, 0x00020000);
#pragma unroll
    for (int j = 0; j < PW; ++j) gr_to_lds_nt(rs, smem + b * BUF + (wave * PW + j) * 1024, wo[j], (t0 + kw) * 128);
    ++sw;
    kw = kw + 1 == n ? 0 : kw + 1;
  };
  const auto load_x = [&](int b) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)X, (short)0, sx < n ? xbytes : 0, 0x00020000);
#pragma unroll
    for (int j = 0; j < PX; ++j) gr_to_lds(rs, smem + b * BUF + XAT + (wave * PX + j) * 1024, xo[j], (t0 + kx) * 128);
    ++sx;
    kx = kx + 1 == n ? 0 : kx + 1;
  };
  f32x4 acc[NI][FR];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int f = 0; f < FR; ++f) acc[i][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 wa[NI], wb[NI], xa[FR], xb[FR];
  __shared__ __attribute__((aligned(16))) bf16 rows[NORM ? LN_ROWS * LN_K : 8];   // NORM: the normalised rows (lanes of other rows read the last)
  __shared__ float sums[NORM ? LN_ROWS * LN_WAVES : 1];
  const char* xrow = reinterpret_cast<const char*>(rows) + min(fr, M - 1) * (LN_K * 2) + 16 * fc;
  int kr = tile % n;   // K tile of the buffer that is read
  const auto read = [&](bf16x8 (&w)[NI], bf16x8 (&x)[FR], int b, int kk) {
    if constexpr (NORM) x[0] = *reinterpret_cast<const bf16x8*>(xrow + kr * 128 + 64 * kk);
    const char* L = smem + b * BUF + 16 * gr_swz(fr, 4 * kk + fc) + fr * 128;
#pragma unroll
    for (int i = 0; i < NI; ++i) w[i] = *reinterpret_cast<const bf16x8*>(L + (wn * NI + i) * 2048);
#pragma unroll
    for (int f = 0; f < (NORM ? 0 : FR); ++f) x[f] = *reinterpret_cast<const bf16x8*>(L + XAT + (wm * FR + f) * 2048);
  };
  const auto mm = [&](const bf16x8 (&w)[NI], const bf16x8 (&x)[FR]) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int f = 0; f < FR; ++f) acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[f], acc[i][f], 0, 0, 0);
  };
  const auto interleave = [&](auto nv_tag) {
    constexpr int NV = decltype(nv_tag)::value;
#pragma unroll
    for (int q = 0; q < NI * FR; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (q < NI + FR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (q < NV) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
  };
  constexpr int CH = LN_K / 8 / (64 * NW);   // NORM: pieces of eight a thread and row
  bf16x8 raw[NORM ? LN_ROWS : 1][CH], gain[CH];
  if constexpr (NORM) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int k = min(8 * (tid + 64 * NW * c), 64 * steps - 8);   // (no branch: the weights' moves would wait for what it loads)
#pragma unroll
      for (int m = 0; m < LN_ROWS; ++m) raw[m][c] = ld8(X + min(m, M - 1) * ldx + k);
      gain[c] = ld8(ln + k);
    }
  }
#pragma unroll
  for (int b = 0; b < NST; ++b) {
    load_w(b);
    if (b < NST - 1) load_x(b);
  }
  if constexpr (NORM) {
#pragma unroll
    for (int m = 0; m < LN_ROWS; ++m) {
      if (m >= M) break;
      float ss[LN_WAVES / NW];   // (of waves wave + NW p of those eight)
#pragma unroll
      for (int p = 0; p < LN_WAVES / NW; ++p) {
        ss[p] = 0.f;
#pragma unroll
        for (int c = p; c < CH; c += LN_WAVES / NW)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float f = (float)raw[m][c][j], next = ss[p] + f * f;
            ss[p] = 8 * (tid + 64 * NW * c) < 64 * steps ? next : ss[p];
          }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int p = 0; p < LN_WAVES / NW; ++p) ss[p] += __shfl_xor(ss[p], o);
#pragma unroll
      for (int p = 0; p < LN_WAVES / NW; ++p)
        if (lane == 0) sums[m * LN_WAVES + wave + NW * p] = ss[p];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int m = 0; m < LN_ROWS; ++m) {
      if (m >= M) break;
      float ss = 0.f;
#pragma unroll
      for (int x = 0; x < LN_WAVES; ++x) ss += sums[m * LN_WAVES + x];
      const float rms = rsqrtf(ss / (float)(64 * steps) + eps);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int k = 8 * (tid + 64 * NW * c);
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (bf16)((float)raw[m][c][j] * rms * (float)gain[c][j]);
        if (k < 64 * steps) *reinterpret_cast<bf16x8*>(rows + m * LN_K + k) = v;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the barrier follows)
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NST - 1) * LPT - PX) : "memory");
  read(wa, xa, 0, 0);
  int b = 0, pb = NST - 1;
  for (int i = 0; i < n; ++i) {
    const int nb = b + 1 == NST ? 0 : b + 1;
    mm(wa, xa);
    read(wb, xb, b, 1);
    kr = kr + 1 == n ? 0 : kr + 1;
    load_x(pb);
    interleave(std::integral_constant<int, PX>{});
    // this wave's moves of the next tile are done (those of NST - 2 tiles are younger) and its reads of this one: the barrier
    // publishes the one and frees the other
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 2) * LPT) : "memory");
    mm(wb, xb);
    read(wa, xa, nb, 0);
    load_w(b);
    interleave(std::integral_constant<int, PW>{});
    pb = b;
    b = nb;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the empty moves past n)

  // D rows are W rows: lane (fr, fc) holds X row fr, columns 4 fc .. + 3 of each block of 16
#pragma unroll
  for (int f = 0; f < FR; ++f) {
    const int row = 16 * (FR * wm + f) + fr, c0 = n0 + wn * NI * 16;
    if (row >= M) continue;
    if constexpr (EPI == GR_PART) {
      float* o = part + ((int64_t)sp * M + row) * N + c0 + 4 * fc;
#pragma unroll
      for (int i = 0; i < NI; ++i) *reinterpret_cast<f32x4*>(o + 16 * i) = acc[i][f];
    } else if constexpr (EPI == GR_SILU) {
      bf16* o = out + row * ldo + c0 / 2 + 4 * fc;
#pragma unroll
      for (int i = 0; i < NI; i += 2) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = acc[i][f][e];
          v[e] = (bf16)(g / (1.f + __expf(-g)) * acc[i + 1][f][e]);
        }
        *reinterpret_cast<bf16x4*>(o + 8 * i) = v;
      }
    } else {
      bf16* o = out + row * ldo + c0 + 4 * fc;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)(acc[i][f][e] + (bias ? (float)bias[c0 + 16 * i + 4 * fc + e] : 0.f));
        *reinterpret_cast<bf16x4*>(o + 16 * i) = v;
      }
    }
  }
}

template <int WM, int WN, int FR, int NST, int EPI, bool NORM = false>
int gr_launch(const bf16* x, int64_t ldx, const bf16* w, int64_t ldw, const bf16* bias, bf16* out, int64_t ldo, int M, int N, int K,
              int splits, float* part, hipStream_t stream, const bf16* ln = nullptr, float eps = 0.f) {
  constexpr int LDS = NST * (BN + (NORM ? 0 : 16 * FR * WM)) * 128;
  const auto kern = gemm_rows_kernel<WM, WN, FR, NST, EPI, NORM>;
  static const hipError_t set = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (set != hipSuccess) return (int)set;
  kern<<<N / BN * splits, 64 * WM * WN, LDS, stream>>>(x, ldx, w, ldw, bias, out, ldo, M, N, K / 64, splits, part, ln, eps);
  OME_CHECK_LAUNCH();
  return 0;
}

template <int EPI>
int gr_rows(const bf16* x, int64_t ldx, const bf16* w, int64_t ldw, const bf16* bias, bf16* out, int64_t ldo, int M, int N, int K,
            int splits, float* part, hipStream_t stream) {
  if (M <= 32) return gr_launch<1, 4, 2, 4, EPI>(x, ldx, w, ldw, bias, out, ldo, M, N, K, splits, part, stream);
  if (M <= 64) return gr_launch<4, 1, 1, 4, EPI>(x, ldx, w, ldw, bias, out, ldo, M, N, K, splits, part, stream);
  // (eight waves of 32 x 64: 46 / 27 / 12 us of the three above; of 64 x 32 48 / 28 / 14)
  if (M <= 128) return gr_launch<4, 2, 2, 5, EPI>(x, ldx, w, ldw, bias, out, ldo, M, N, K, splits, part, stream);
  // (eight waves of 32 x 128: 60 / 37 us of the first two; of 64 x 64 66 / 39, four of 128 x 64 83 / 46, sixteen of 64 x 32 66 / 40)
  return gr_launch<8, 1, 2, 3, EPI>(x, ldx, w, ldw, bias, out, ldo, M, N, K, splits, part, stream);
}

}  // namespace

// epi 0: out = x w^T (+ bias), 2: SiLU(gate) * up of weights interleaved in blocks of 16 rows (out is N / 2 wide), both one split;
// 3: part[splits][M][N] = the fp32 sums over each piece of K.  -3: operands that the kernel does not take (nothing is launched).
OME_API int ome_gemm_rows(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, void* out, int64_t ldo, int M,
                          int N, int K, int epi, int splits, float* part, hipStream_t stream) {
  if (M <= 0 || M > 256 || N <= 0 || N % BN || K < 64 || K % 64 || splits < 1 || splits > K / 64 || ldx < K || ldw < K || ldx % 8 || ldw % 8 ||
      (uintptr_t)x % 16 || (uintptr_t)w % 16 || 2 * 256 * ldx > 0x7fffffff || 2 * BN * ldw > 0x7fffffff ||
      (int64_t)(N / BN) * splits > 0x7fffffff)
    return -3;
  if (epi == GR_PART ? !part || (uintptr_t)part % 16 : !out || splits != 1 || ldo % 4 || (uintptr_t)out % 8) return -3;
  const auto run = epi == GR_BF16 ? gr_rows<GR_BF16> : epi == GR_SILU ? gr_rows<GR_SILU> : epi == GR_PART ? gr_rows<GR_PART> : nullptr;
  return run ? run((const bf16*)x, ldx, (const bf16*)w, ldw, (const bf16*)bias, (bf16*)out, ldo, M, N, K, splits, part, stream) : -3;
}

// out = SiLU(gate) * up of RMSNorm(x) w^T (norm weights ln [K]), w interleaved as for epi 2 above; one or two rows.  -3 as above.
OME_API int ome_gemm_rows_norm(const void* x, int64_t ldx, const void* ln, float eps, const void* w, int64_t ldw, void* out, int64_t ldo, int M, int N,
                               int K, hipStream_t stream) {
  if (M <= 0 || M > LN_ROWS || N <= 0 || N % BN || K < 64 || K > LN_K || K % 64 || ldx < K || ldw < K || ldx % 8 || ldw % 8 || ldo % 4 || !out ||
      ((uintptr_t)x | (uintptr_t)w | (uintptr_t)ln) % 16 || (uintptr_t)out % 8 || 2 * BN * ldw > 0x7fffffff)
    return -3;
  return gr_launch<1, 4, 1, 5, GR_SILU, true>((const bf16*)x, ldx, (const bf16*)w, ldw, nullptr, (bf16*)out, ldo, M, N, K, 1, nullptr, stream,
                                              (const bf16*)ln, eps);
}
