// Mixture-of-Experts kernels (SURVEY.md §2.9 K10 routing + K11 grouped GEMM) for gfx950.
//
//   ome_moe_route   : gate logits [T, E] -> softmax (or sigmoid) -> top-k ids / weights,
//                     optional renormalisation; one wave per token, E <= 512, k <= 16.
//   ome_moe_align   : counting sort of the T*k assignments by expert -> expert_offsets [E+1],
//                     sorted_ids [T*k] (flat assignment index t*k+j) and its inverse, all on the
//                     device (graph-capturable: no host sync on the per-expert counts).
//   ome_moe_gemm    : grouped GEMM  out[p, :] = A[row(p), :] @ W[e(p)]^T  over the sorted
//                     assignments p; A rows are gathered through sorted_ids / k (gate_up) or
//                     read in sorted order (down).  Tiles never straddle experts; each workgroup finds its
//                     (expert, m-tile) by scanning the offsets, so the grid is a static upper bound.
//   ome_moe_gemm_stream : the same for experts with few rows, on tiles listed by ome_moe_align_tiles
//   ome_moe_combine : out[t] = sum_j w[t, j] * Y[inv[t*k + j]]   (fp32 accumulate)
#include "common.h"

#include <type_traits>
#include "lds_stages.h"

#include <cstdlib>

#ifndef OME_NEG_INF
#define OME_NEG_INF (-__builtin_inff())
#endif

// ------------------------------------------------------------------------------------------
// routing
// ------------------------------------------------------------------------------------------
// group_mode: 0 = plain top-k; 1 = DeepSeek-V2 "group_limited_greedy" (group score = max);
// 2 = DeepSeek-V3 "noaux_tc" (group score = sum of the group's top-2 biased scores).  Experts are
// chosen on score + bias (``e_score_correction_bias``) restricted to the best ``topk_group``
// groups (other experts score 0, as in the HF reference); weights are the unbiased scores.
// 3 = group score = max like 1, but experts outside the chosen groups count as minus infinity (never
// chosen while an allowed expert is left, however negative the biased scores are); 4 = group score
// like 2, exclusion like 3.
//
// One wave per token, expert lane + 64 i in register i of NV.  A pick is one maximum over the wave of (key as
// an ordered integer, lowest expert first), five vector instructions a level through DPP and the permlane
// swaps; three shuffles a level through LDS, and picks written and rescaled in memory one by one, took 20 us for 48
// tokens of 512 experts top 10 (now 12).
template <int C>
__device__ __forceinline__ uint64_t dpp_max(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, C, 0xF, 0xF, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), C, 0xF, 0xF, false);
  const uint64_t o = (uint64_t)hi << 32 | lo;
  return o > v ? o : v;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
  v = dpp_max<0xB1>(v);    // quad_perm: lane ^ 1
  v = dpp_max<0x4E>(v);    // quad_perm: lane ^ 2
  v = dpp_max<0x141>(v);   // row_half_mirror: the other four of eight
  v = dpp_max<0x140>(v);   // row_mirror: the other eight of sixteen
  const auto l = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
  const uint64_t a = (uint64_t)h[0] << 32 | l[0], b = (uint64_t)h[1] << 32 | l[1];
  v = a > b ? a : b;
  const auto l2 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  const auto h2 = __builtin_amdgcn_permlane32_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
  const uint64_t c = (uint64_t)h2[0] << 32 | l2[0], d = (uint64_t)h2[1] << 32 | l2[1];
  return c > d ? c : d;
}
// keys in order as unsigned integers above 0 (-0 = +0); 0: NaN, never picked
__device__ __forceinline__ uint32_t ordered_key(float x) {
  const uint32_t u = __float_as_uint(x + 0.f);
  return x != x ? 0u : u & 0x80000000u ? ~u : u | 0x80000000u;
}

template <typename T, int MAXV>
__global__ __launch_bounds__(256) void moe_route_kernel(const T* __restrict__ logits, int64_t stride, int n_tok,
                                                        int E, int k, int renorm, int scoring,
                                                        const float* __restrict__ bias, int n_group, int topk_group,
                                                        int group_mode, float* __restrict__ topk_w,
                                                        int* __restrict__ topk_ids,
                                                        const float* __restrict__ logit_bias) {
  __shared__ float s_key[4][512];
  __shared__ int s_gsel[4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + wave;
  if (t >= n_tok) return;
  float v[MAXV], key[MAXV];   // E <= 64 MAXV
  const T* row = logits + (int64_t)t * stride;
  float mx = OME_NEG_INF;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int e = lane + 64 * i;
    // (logit_bias: a router bias that is part of the logits, so it counts in the scores and weights)
    v[i] = e < E ? (float)row[e] + (logit_bias ? logit_bias[e] : 0.f) : OME_NEG_INF;
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int e = lane + 64 * i;
    float p;
    if (scoring == 0) p = e < E ? __expf(v[i] - mx) : 0.f;        // softmax numerator
    else p = e < E ? 1.f / (1.f + __expf(-v[i])) : -1.f;           // sigmoid score
    v[i] = p;
    sum += (e < E && scoring == 0) ? p : 0.f;
  }
  if (scoring == 0) {
    sum = wave_sum(sum);
    const float inv = 1.f / sum;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) v[i] *= inv;
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int e = lane + 64 * i;
    key[i] = e < E ? v[i] + (bias ? bias[e] : 0.f) : OME_NEG_INF;
  }
  if (group_mode && n_group > 1) {
    const int gs = E / n_group;
#pragma unroll
    for (int i = 0; i < MAXV; ++i)
      if (lane + 64 * i < E) s_key[wave][lane + 64 * i] = key[i];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    float gscore = OME_NEG_INF;
    if (lane < n_group) {
      float b1 = OME_NEG_INF, b2 = OME_NEG_INF;
      for (int j = 0; j < gs; ++j) {
        const float x = s_key[wave][lane * gs + j];
        if (x > b1) {
          b2 = b1;
          b1 = x;
        } else if (x > b2) {
          b2 = x;
        }
      }
      gscore = group_mode == 2 || group_mode == 4 ? b1 + (gs > 1 ? b2 : 0.f) : b1;
    }
    int chosen = 0;  // bit set on the lanes whose group is selected
    for (int j = 0; j < topk_group; ++j) {
      float best = gscore;
      int bi = lane < n_group ? lane : 1 << 30;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o);
        const int oi = __shfl_xor(bi, o);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (lane == bi) {
        chosen = 1;
        gscore = OME_NEG_INF;
      }
    }
    s_gsel[wave][lane] = chosen;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int e = lane + 64 * i;
      if (e < E && !s_gsel[wave][e / gs]) key[i] = group_mode >= 3 ? OME_NEG_INF : 0.f;
    }
  }
  float picked_sum = 0.f, my_w = 0.f;
  int my_id = 0;   // lane j keeps pick j
  uint64_t cand[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int e = lane + 64 * i;
    const uint32_t o = e < E ? ordered_key(key[i]) : 0u;
    cand[i] = o ? (uint64_t)o << 32 | (uint32_t)~e : 0ull;   // (ties -> lowest expert id)
  }
  for (int j = 0; j < k; ++j) {
    // keys may be any value or an infinity (masked groups: -inf)
    uint64_t best = cand[0];
#pragma unroll
    for (int i = 1; i < MAXV; ++i) best = cand[i] > best ? cand[i] : best;
    best = wave_max_u64(best);
    int bi = __builtin_amdgcn_readfirstlane((int)~(uint32_t)best);
    float bw = 0.f;
    if (__builtin_amdgcn_readfirstlane((uint32_t)(best >> 32)) == 0) {
      bi = j < E ? j : E - 1;   // no key beat the floor (NaN logits): still emit a valid expert id
    } else {
      float at = v[0];
#pragma unroll
      for (int i = 1; i < MAXV; ++i) at = (bi >> 6) == i ? v[i] : at;
      bw = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(at), bi & 63));
    }
    if (k > 64 && lane == 0) {
      topk_w[(int64_t)t * k + j] = bw;
      topk_ids[(int64_t)t * k + j] = bi;
    }
    if (lane == j) my_w = bw, my_id = bi;
    picked_sum += bw;
#pragma unroll
    for (int i = 0; i < MAXV; ++i)  // remove the winner (static register indexing)
      if (lane + 64 * i == bi) cand[i] = 0ull;
  }
  const float inv = renorm ? 1.f / (picked_sum + 1e-20f) : 1.f;
  if (k <= 64) {
    if (lane < k) {
      topk_w[(int64_t)t * k + lane] = renorm ? my_w * inv : my_w;
      topk_ids[(int64_t)t * k + lane] = my_id;
    }
  } else if (renorm && lane == 0) {
    for (int j = 0; j < k; ++j) topk_w[(int64_t)t * k + j] *= inv;
  }
}

OME_API int ome_moe_route(const void* logits, int is_bf16, int64_t stride, int n_tok, int E, int k, int renorm,
                          int scoring, const float* bias, int n_group, int topk_group, int group_mode,
                          float* topk_w, int* topk_ids, const float* logit_bias, hipStream_t stream) {
  if (n_tok <= 0) return 0;
  if (E > 512 || k > E || k <= 0) return -2;
  if (group_mode && n_group > 1 && (E % n_group || n_group > 64 || topk_group > n_group)) return -2;
  const int g = (n_tok + 3) / 4;
#define ROUTE(T, NV)                                                                                                   \
  moe_route_kernel<T, NV><<<g, 256, 0, stream>>>((const T*)logits, stride, n_tok, E, k, renorm, scoring, bias, n_group, \
                                                 topk_group, group_mode, topk_w, topk_ids, logit_bias)
  if (is_bf16) {
    if (E <= 64) ROUTE(bf16, 1);
    else if (E <= 128) ROUTE(bf16, 2);
    else if (E <= 256) ROUTE(bf16, 4);
    else ROUTE(bf16, 8);
  } else {
    if (E <= 64) ROUTE(float, 1);
    else if (E <= 128) ROUTE(float, 2);
    else if (E <= 256) ROUTE(float, 4);
    else ROUTE(float, 8);
  }
#undef ROUTE
  OME_CHECK_LAUNCH();
  return 0;
}

// ------------------------------------------------------------------------------------------
// alignment (counting sort by expert), single workgroup
// Bound by one CU: a store to a place of its own for every assignment, and two round trips for every 1024 of them.  Up to 32 a thread are read eight at a
// time and stay in registers, with the place among their expert's that counting them returns, and are put in order in LDS, from where they leave in
// rows: us, 30000 assignments of 512 experts 25.9 -> 10.9, 15000 14.5 -> 7.7, 4000 6.2 -> 5.5, 18000 of 128 15.1 -> 8.4, 5600 of 256 7.3 -> 5.7, 6000 of 8 7.1 ->
// 6.7.  Fewer take the two passes: 480 3.8 -> 4.9, 2400 of 128 4.9 -> 5.1.
// ------------------------------------------------------------------------------------------
constexpr int ALIGN_KEEP = 32, ALIGN_AT_ONCE = 8;
constexpr bool align_keeps(int n) { return n > 3072 && n <= ALIGN_KEEP * 1024; }

__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ topk_ids, int n, int E,
                                                         int* __restrict__ offsets, int* __restrict__ sorted_ids,
                                                         int* __restrict__ inv, int4* __restrict__ tiles, int bm, int e_tiles,
                                                         int max_tiles) {
  extern __shared__ int sh[];  // [E] counts, [E] cursors, [n] assignments in order where threads keep them (n < 2^16)
  int* cnt = sh;
  int* cur = sh + E;
  for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  // ids outside [0, E) (never produced by moe_route) are clamped rather than indexing LDS out of range
  const bool keep = align_keeps(n);   // (counts of E experts in LDS: E < 2^16)
  uint32_t kept[ALIGN_KEEP];   // expert << 16 | place
  if (keep) {
#pragma unroll
    for (int b = 0; b < ALIGN_KEEP; b += ALIGN_AT_ONCE) {
      if (b * 1024 >= n) continue;   // whole block
      int id[ALIGN_AT_ONCE];
#pragma unroll
      for (int u = 0; u < ALIGN_AT_ONCE; ++u)
        if ((b + u) * 1024 < n) id[u] = topk_ids[min((b + u) * 1024 + (int)threadIdx.x, n - 1)];
#pragma unroll
      for (int u = 0; u < ALIGN_AT_ONCE; ++u)
        if ((b + u) * 1024 + (int)threadIdx.x < n) {
          const int e = min(max(id[u], 0), E - 1);
          kept[b + u] = (uint32_t)e << 16 | (uint32_t)atomicAdd(&cnt[e], 1);
        }
    }
  } else {
    for (int i = threadIdx.x; i < n; i += blockDim.x) atomicAdd(&cnt[min(max(topk_ids[i], 0), E - 1)], 1);
  }
  __syncthreads();
  // exclusive prefix sums: a thread's run of experts, its wave, the waves before (one thread summing 512 experts
  // through LDS took 15 of the kernel's 20 us)
  __shared__ int s_wave[16], s_tiles[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, per = (E + 1023) / 1024, e0 = threadIdx.x * per;
  int own = 0, own_t = 0;
  for (int i = 0; i < per; ++i)
    if (e0 + i < E) {
      own += cnt[e0 + i];
      own_t += e0 + i < e_tiles ? (cnt[e0 + i] + bm - 1) / bm : 0;
    }
  int incl = own, incl_t = own_t;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(incl, d), up_t = __shfl_up(incl_t, d);
    if (lane >= d) {
      incl += up;
      incl_t += up_t;
    }
  }
  if (lane == 63) {
    s_wave[wave] = incl;
    s_tiles[wave] = incl_t;
  }
  __syncthreads();
  int acc = incl - own, t = incl_t - own_t;
  for (int w = 0; w < wave; ++w) {
    acc += s_wave[w];
    t += s_tiles[w];
  }
  for (int i = 0; i < per; ++i)
    if (e0 + i < E) {
      offsets[e0 + i] = acc;
      cur[e0 + i] = acc;
      const int end = acc + cnt[e0 + i];
      if (e0 + i < e_tiles)
        for (int m = acc; m < end; m += bm, ++t)
          if (t < max_tiles) tiles[t] = int4{e0 + i, m, end, 0};
      acc = end;
    }
  if (threadIdx.x == 1023) offsets[E] = acc;   // (its run is the last, or empty: the total)
  if (tiles != nullptr) {   // the rest have no expert, but the number of those that have
    int all = 0;
    for (int w = 0; w < 16; ++w) all += s_tiles[w];
    for (int i = all + threadIdx.x; i < max_tiles; i += blockDim.x) tiles[i] = int4{-1, 0, 0, all};
  }
  __syncthreads();
  // stable within an expert is not required (the combine uses the inverse map)
  if (keep) {
    uint16_t* const order = reinterpret_cast<uint16_t*>(sh + 2 * E);
#pragma unroll
    for (int b = 0; b < ALIGN_KEEP; ++b) {
      const int i = b * 1024 + threadIdx.x;
      if (i < n) {
        const int p = cur[kept[b] >> 16] + (int)(kept[b] & 0xffff);
        order[p] = (uint16_t)i;
        inv[i] = p;
      }
    }
    __syncthreads();
    for (int p = threadIdx.x; p < n; p += 1024) sorted_ids[p] = order[p];
    return;
  }
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int p = atomicAdd(&cur[min(max(topk_ids[i], 0), E - 1)], 1);
    sorted_ids[p] = i;
    inv[i] = p;
  }
}

static int align_launch(const int* topk_ids, int n, int E, int* offsets, int* sorted_ids, int* inv, int4* tiles, int bm, int e_tiles, int max_tiles,
                        hipStream_t stream) {
  constexpr int MOST = 128 << 10;
  const int lds = 2 * E * (int)sizeof(int) + (align_keeps(n) ? 2 * n : 0);
  static const hipError_t set = hipFuncSetAttribute((const void*)moe_align_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MOST);
  if (lds > 64 << 10 && (set != hipSuccess || lds > MOST)) return -2;
  moe_align_kernel<<<1, 1024, lds, stream>>>(topk_ids, n, E, offsets, sorted_ids, inv, tiles, bm, e_tiles, max_tiles);
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_moe_align(const int* topk_ids, int n, int E, int* offsets, int* sorted_ids, int* inv,
                          hipStream_t stream) {
  if (n <= 0) {
    return hipMemsetAsync(offsets, 0, (E + 1) * sizeof(int), stream);
  }
  return align_launch(topk_ids, n, E, offsets, sorted_ids, inv, nullptr, 1, 0, 0, stream);
}

// ... and the tiles of `bm` rows of one expert each, of experts below `e_tiles`, (expert, first row, the expert's end, 0), 16-byte aligned: a workgroup of the
// kernels below reads its own instead of searching the offsets (512 experts: eight rounds of a wave's prefix sum, 2 us a
// workgroup).  max_tiles >= min(n, E) + n / bm bounds their number; entries past it have expert -1 and that number in the last place.
OME_API int ome_moe_align_tiles(const int* topk_ids, int n, int E, int* offsets, int* sorted_ids, int* inv, int* tiles, int bm,
                                int e_tiles, int max_tiles, hipStream_t stream) {
  if (n <= 0 || bm <= 0 || max_tiles < (n < E ? n : E) + n / bm || (uintptr_t)tiles % 16) return -2;
  return align_launch(topk_ids, n, E, offsets, sorted_ids, inv, (int4*)tiles, bm, e_tiles, max_tiles, stream);
}

// ------------------------------------------------------------------------------------------
// grouped GEMM: 64x64 output tile per 256-thread workgroup, BK = 32, MFMA 16x16x32 bf16.
// Waves as 2(M) x 2(N), each 32x32 = 2x2 MFMA tiles.  LDS rows padded to 40 bf16 (80 B) so
// the 16 rows a ds_read_b128 group touches start on distinct bank quads.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int GBM = 64, GBN = 64, GBK = 32, GLD = GBK + 8;

__global__ __launch_bounds__(256) void moe_gemm_kernel(const bf16* __restrict__ A, int64_t lda,
                                                       const int* __restrict__ sorted_ids, int gather_div,
                                                       const bf16* __restrict__ W, const int* __restrict__ offsets,
                                                       int E, int N, int K, bf16* __restrict__ out, int64_t ldo,
                                                       const bf16* __restrict__ bias) {
  __shared__ __attribute__((aligned(16))) bf16 sA[GBM * GLD];
  __shared__ __attribute__((aligned(16))) bf16 sB[GBN * GLD];
  __shared__ int s_tile[3];
  // ---- find (expert, m0) of this workgroup's tile ----
  if (threadIdx.x == 0) {
    int t = blockIdx.y, e = 0, found = 0;
    for (; e < E; ++e) {
      const int c = offsets[e + 1] - offsets[e];
      const int nt = (c + GBM - 1) / GBM;
      if (t < nt) {
        found = 1;
        break;
      }
      t -= nt;
    }
    s_tile[0] = found ? e : -1;
    s_tile[1] = found ? offsets[e] + t * GBM : 0;
    s_tile[2] = found ? offsets[e + 1] : 0;
  }
  __syncthreads();
  const int e = s_tile[0];
  if (e < 0) return;
  const int m0 = s_tile[1], m_end = s_tile[2];
  const int n0 = blockIdx.x * GBN;
  const bf16* We = W + (int64_t)e * N * K;

  const int tid = threadIdx.x;
  // global->LDS staging: each thread moves one 16-B chunk of A and one of B per k-step
  const int lr = tid >> 2, lc = (tid & 3) * 8;  // row 0..63, k offset 0/8/16/24
  const int arow = m0 + lr;
  int64_t a_off = -1;
  if (arow < m_end) {
    const int src = gather_div > 0 ? sorted_ids[arow] / gather_div : arow;
    a_off = (int64_t)src * lda;
  }
  const int brow = n0 + lr;
  const bf16* bptr = brow < N ? We + (int64_t)brow * K : nullptr;

  const int wave = tid >> 6, lane = tid & 63;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16x8 ra = {}, rb = {};
  if (a_off >= 0) ra = ld8(A + a_off + lc);
  if (bptr) rb = ld8(bptr + lc);
  for (int k0 = 0; k0 < K; k0 += GBK) {
    __syncthreads();
    *reinterpret_cast<bf16x8*>(&sA[lr * GLD + lc]) = ra;
    *reinterpret_cast<bf16x8*>(&sB[lr * GLD + lc]) = rb;
    __syncthreads();
    if (k0 + GBK < K) {  // prefetch the next k-step while this one computes
      if (a_off >= 0) ra = ld8(A + a_off + k0 + GBK + lc);
      if (bptr) rb = ld8(bptr + k0 + GBK + lc);
    }
    bf16x8 af[2], bfr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) af[i] = *reinterpret_cast<const bf16x8*>(&sA[(wm + 16 * i + fr) * GLD + fk]);
#pragma unroll
    for (int j = 0; j < 2; ++j) bfr[j] = *reinterpret_cast<const bf16x8*>(&sB[(wn + 16 * j + fr) * GLD + fk]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
  }
  // ---- epilogue: C lane map row = 4*(l>>4)+r, col = l&15 ----
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int col = n0 + wn + 16 * j + (lane & 15);
        if (row < m_end && col < N) {
          const float b = bias != nullptr ? (float)bias[(int64_t)e * N + col] : 0.f;  // per-expert bias (GPT-OSS)
          out[(int64_t)row * ldo + col] = (bf16)(acc[i][j][r] + b);
        }
      }
}

// ------------------------------------------------------------------------------------------
// grouped GEMM v2: 128 x 128 tiles, 2x2 waves, a BK k-step staged through DOUBLE-buffered LDS: the next step's global
// loads are issued before this step's MFMAs and written to the other buffer after them, so one barrier per k-step.  Some 60 rows
// per expert and more (fewer: moe_stream_kernel; 46 and more, and shapes that its tiles take: gemm_pp.hip).
// ------------------------------------------------------------------------------------------
template <int BM, int BN, int BK>
__global__ __launch_bounds__(256) void moe_gemm_v2_kernel(const bf16* __restrict__ A, int64_t lda,
                                                          const int* __restrict__ sorted_ids, int gather_div,
                                                          const bf16* __restrict__ W, const int* __restrict__ offsets,
                                                          int E, int N, int K, bf16* __restrict__ out, int64_t ldo,
                                                          const bf16* __restrict__ bias) {
  constexpr int LD = BK + 8, CPR = BK / 8;           // padded LDS row, 16-B chunks per row
  constexpr int CA = BM * CPR / 256, CB = BN * CPR / 256;  // chunks per thread per operand
  constexpr int MI = BM / 32, NJ = BN / 32;          // 16x16 MFMA tiles per wave (waves 2 x 2)
  static_assert(CA >= 1 && CB >= 1 && 2 * (BM + BN) * LD * 2 <= 65536, "tile");
  __shared__ __attribute__((aligned(16))) bf16 smem[2 * (BM + BN) * LD];
  __shared__ int s_tile[3];
  bf16* sA = smem;                  // [2][BM * LD]
  bf16* sB = smem + 2 * BM * LD;    // [2][BN * LD]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // ---- (expert, m0) of this tile: wave 0 prefix-sums the per-expert tile counts 64 at a time ----
  if (tid == 0) s_tile[0] = -1;
  __syncthreads();
  if (wave == 0) {
    int base = 0;
    const int y = blockIdx.y;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const int nt = e < E ? (offsets[e + 1] - offsets[e] + BM - 1) / BM : 0;
      int incl = nt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d);
        if (lane >= d) incl += v;
      }
      const int t = y - base;
      if (t >= incl - nt && t < incl) {
        s_tile[0] = e;
        s_tile[1] = offsets[e] + (t - (incl - nt)) * BM;
        s_tile[2] = offsets[e + 1];
      }
      base += __shfl(incl, 63);
      if (y < base) break;
    }
  }
  __syncthreads();
  const int e = s_tile[0];
  if (e < 0) return;
  const int m0 = s_tile[1], m_end = s_tile[2];
  const int n0 = blockIdx.x * BN;
  const bf16* We = W + (int64_t)e * N * K;
  const int lc = (tid % CPR) * 8;
  int64_t a_off[CA];
  const bf16* bptr[CB];
#pragma unroll
  for (int j = 0; j < CA; ++j) {
    const int arow = m0 + (tid + 256 * j) / CPR;
    a_off[j] = -1;
    if (arow < m_end) a_off[j] = (int64_t)(gather_div > 0 ? sorted_ids[arow] / gather_div : arow) * lda;
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int r = n0 + (tid + 256 * j) / CPR;
    bptr[j] = r < N ? We + (int64_t)r * K : nullptr;
  }
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  f32x4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16x8 ra[CA], rb[CB];
  auto gload = [&](int k0) {
#pragma unroll
    for (int j = 0; j < CA; ++j) ra[j] = a_off[j] >= 0 ? ld8(A + a_off[j] + k0 + lc) : bf16x8{};
#pragma unroll
    for (int j = 0; j < CB; ++j) rb[j] = bptr[j] ? ld8(bptr[j] + k0 + lc) : bf16x8{};
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int j = 0; j < CA; ++j)
      *reinterpret_cast<bf16x8*>(&sA[buf * BM * LD + ((tid + 256 * j) / CPR) * LD + lc]) = ra[j];
#pragma unroll
    for (int j = 0; j < CB; ++j)
      *reinterpret_cast<bf16x8*>(&sB[buf * BN * LD + ((tid + 256 * j) / CPR) * LD + lc]) = rb[j];
  };
  const int nk = K / BK;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int ks = 0; ks < nk; ++ks) {
    const int cur = ks & 1;
    if (ks + 1 < nk) gload((ks + 1) * BK);  // in flight during this step's MFMAs
    const bf16* a_s = sA + cur * BM * LD;
    const bf16* b_s = sB + cur * BN * LD;
#pragma unroll
    for (int kk = 0; kk < BK; kk += 32) {
      bf16x8 af[MI], bfr[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = *reinterpret_cast<const bf16x8*>(&a_s[(wm + 16 * i + fr) * LD + kk + fk]);
#pragma unroll
      for (int j = 0; j < NJ; ++j) bfr[j] = *reinterpret_cast<const bf16x8*>(&b_s[(wn + 16 * j + fr) * LD + kk + fk]);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
    }
    if (ks + 1 < nk) lstore(cur ^ 1);  // the other buffer was last read before the previous barrier
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int col = n0 + wn + 16 * j + (lane & 15);
        if (row < m_end && col < N) {
          const float b = bias != nullptr ? (float)bias[(int64_t)e * N + col] : 0.f;
          out[(int64_t)row * ldo + col] = (bf16)(acc[i][j][r] + b);
        }
      }
}


// ------------------------------------------------------------------------------------------
// bf16 experts with few rows each: out[p, :] = A[row(p)] . W[e(p)]^T (+ bias) over 64-row tiles, one workgroup per tile and 64 weight
// rows.  Bound by the weights' way from memory: three (few workgroups: four) stages of 64 k move to LDS by DMA (lds_stages.h: one stage
// before the wait, two or three behind it); a workgroup reads its tile instead of searching it.  A wave without rows of its own only moves.
// 128 weight rows a workgroup: half as many and twice as long, 3 to 5% slower with 2048 or fewer k and 1 to 3% faster with 2688.
// Whole layer, us (register-staged 64 x 64 tiles with the search -> this): 512 experts top 10 of 2048 x 512, 1 / 48 / 1000 rows 110 ->
// 67, 430 -> 330 (5.9 TB/s), 780 -> 645; 8 experts top 2 of 4096 x 14336, 1 / 8 / 136 rows 281 -> 182, 465 -> 398 (6.4 TB/s), 673 ->
// 569; 128 experts top 6 of 2688 x 1856, 7 / 70 / 600 rows 145 -> 139, 335 -> 308, 491 -> 490.
// ------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void moe_lds_t;
typedef __attribute__((address_space(1))) void moe_glb_t;

// This workgroup's place in the grid of (blocks of columns, tiles); a tile past the last: none.  Workgroups go to the XCDs in turn.  With `runs` those of an XCD
// take a run of the tiles, all blocks of each, and so walk through one stretch of the weights.  In the grid's order, where a tile's blocks are a multiple of 8,
// an XCD has every eighth block of every tile, 64 rows at eight times that distance, which memory serves more slowly.  Whole layers, us, 8 experts of 4096 x
// 14336, 1, 4, 16, 64 and 128 rows 180 -> 165, 360 -> 328, 468 -> 428, 528 -> 500, 568 -> 552; 512 of 2048 x 512, 48 and 256 rows 326 -> 310, 557 -> 541.  But runs of
// tiles with many rows are unequal work, and without that multiple there is nothing to gain (128 experts of 2688 x 1856, 400 rows 417 -> 435; 512 experts with 43 rows each
// 774 -> 783; 8 with 45 664 -> 666).
__device__ __forceinline__ int2 xcd_place(const int4* __restrict__ tiles, bool runs) {
  if (!runs) return {(int)blockIdx.x, (int)blockIdx.y};
  const int4 last = tiles[gridDim.y - 1];
  const int n = gridDim.x, all = (last.x < 0 ? last.w : (int)gridDim.y) * n, b = blockIdx.y * n + blockIdx.x;
  if (b >= all) return {0, -1};
  const int xcd = b & 7, q = all >> 3, r = all & 7, id = xcd * q + min(xcd, r) + (b >> 3), t = id / n;
  return {id - t * n, t};
}

// Whether tile t is its expert's only one (of `bm` rows): its weights are read once, so they come with the non-temporal policy, and what is read again (rows,
// the weights of experts with more tiles) stays in the caches.  Whole layers, us: 512 experts of 2048 x 512, 48, 256 and 1000 rows 310 -> 281 (6.9 TB/s), 541 ->
// 490, 636 -> 612; 8 of 4096 x 14336, 4, 16 and 128 rows 330 -> 296, 427 -> 386 (7.3 TB/s), 552 -> 509; 128 of 2688 x 1856, 128 and 400 rows 343 -> 315, 415 ->
// 395; 256 fp8 experts of 7168 x 2048, 16, 128 and 700 rows 577 -> 529, 1303 -> 1210, 1768 -> 1731.  With this policy for experts of more tiles too: 600 rows of
// 128 experts 485 -> 522, 2200 of 512 770 -> 820.  The policy is a constant of a move, so the loop stands twice: a branch at each move cost
// few workgroups up to 15%.
__device__ __forceinline__ bool only_tile(const int4* __restrict__ tiles, int t, const int4& tile, int bm) {
  return tile.z - tile.y <= bm && (t == 0 || tiles[t - 1].x != tile.x);
}
using KeptWeights = std::integral_constant<int, 0>;
using ReadOnce = std::integral_constant<int, 2>;
template <int POLICY>
__device__ __forceinline__ void weights_to_lds(const void* src, char* lds, std::integral_constant<int, POLICY>) {
  __builtin_amdgcn_global_load_lds((moe_glb_t*)src, (moe_lds_t*)lds, 16, 0, POLICY);
}

// 16-byte piece `chunk` of a 128-byte row in LDS: 16 rows' pieces in all banks
__device__ __forceinline__ int mswz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

template <int BM, int BN, int NST, int WM>
__global__ __launch_bounds__(256) void moe_stream_kernel(const bf16* __restrict__ A, int64_t lda, const int* __restrict__ sorted_ids,
                                                         int gather_div, const bf16* __restrict__ W, const int4* __restrict__ tiles,
                                                         int N, int K, bf16* __restrict__ out, int64_t ldo,
                                                         const bf16* __restrict__ bias, bool runs) {
  constexpr int AB = BM * 128, STG = AB + BN * 128;             // a stage: 64 k of BM rows and of BN weight rows
  constexpr int WN = 4 / WM, MJ = BM / 16 / WM, NI = BN / 16 / WN;   // waves, 16 x 16 blocks of a wave
  constexpr int AI = BM / 32, WI = BN / 32;                     // moves of 8 rows of a wave
  __shared__ __attribute__((aligned(16))) char smem[NST * STG];
  const int2 at = xcd_place(tiles, runs);
  if (at.y < 0) return;
  const int4 tile = tiles[at.y];
  const int e = tile.x, m0 = tile.y, m_end = tile.z, n0 = at.x * BN, nt = K / 64;
  const bool once = __builtin_amdgcn_readfirstlane(only_tile(tiles, at.y, tile, BM));
  if (e < 0) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int srow[AI];
#pragma unroll
  for (int j = 0; j < AI; ++j) {
    const int p = min(m0 + (wave * AI + j) * 8 + (lane >> 3), m_end - 1);
    srow[j] = gather_div > 0 ? sorted_ids[p] : p;
  }
#pragma unroll
  for (int j = 0; j < AI; ++j) asm volatile("" ::"v"(srow[j]) : "memory");   // the rows' numbers come before any move: the compiler's wait for them is for all that is out
  const bf16* We = W + (int64_t)e * N * K;
  const bf16 *asrc[AI], *wsrc[WI];
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int r = (wave * WI + j) * 8 + (lane >> 3);
    wsrc[j] = We + (int64_t)min(n0 + r, N - 1) * K + mswz(r, lane & 7) * 8;
  }
#pragma unroll
  for (int j = 0; j < AI; ++j) {
    const int r = (wave * AI + j) * 8 + (lane >> 3);
    asrc[j] = A + (int64_t)(gather_div > 0 ? srow[j] / gather_div : srow[j]) * lda + mswz(r, lane & 7) * 8;
  }
  const auto stage = [&](int buf, int kt, auto policy) {
#pragma unroll
    for (int j = 0; j < WI; ++j)
      weights_to_lds(wsrc[j] + kt * 64, smem + buf * STG + AB + (wave * WI + j) * 1024, policy);
#pragma unroll
    for (int j = 0; j < AI; ++j)
      __builtin_amdgcn_global_load_lds((moe_glb_t*)(asrc[j] + kt * 64), (moe_lds_t*)(smem + buf * STG + (wave * AI + j) * 1024), 16, 0, 0);
  };
  const int wm = wave / WN, wn = wave % WN, fr = lane & 15, fc = lane >> 4;
  const bool works = __builtin_amdgcn_readfirstlane(m0 + wm * MJ * 16 < m_end);   // a wave without rows only moves
  f32x4 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto landed = [](auto out) {
    // every wave's block landed; every wave done reading the one before
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(decltype(out)::value) : "memory");
  };
  const auto multiply = [&](int cur) {
    const char *la = smem + cur * STG, *lw = la + AB;
    if (works) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf16x8 xa[MJ];
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          const int r = (wm * MJ + j) * 16 + fr;
          xa[j] = *reinterpret_cast<const bf16x8*>(la + r * 128 + mswz(r, 4 * kk + fc) * 16);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r = (wn * NI + i) * 16 + fr;
          const bf16x8 wf = *reinterpret_cast<const bf16x8*>(lw + r * 128 + mswz(r, 4 * kk + fc) * 16);
#pragma unroll
          for (int j = 0; j < MJ; ++j) acc[i][j] = mfma16(wf, xa[j], acc[i][j]);
        }
      }
    }
  };
  if (once) lds_stages<NST, AI + WI>(nt, [&](int buf, int kt) { stage(buf, kt, ReadOnce{}); }, landed, multiply);
  else lds_stages<NST, AI + WI>(nt, [&](int buf, int kt) { stage(buf, kt, KeptWeights{}); }, landed, multiply);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the copies of the last block past the end
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int p = m0 + (wm * MJ + j) * 16 + fr;
    if (p >= m_end) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = n0 + (wn * NI + i) * 16 + 4 * fc;
      f32x4 v = acc[i][j];
      if (bias != nullptr)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += (float)bias[(int64_t)e * N + min(n + r, N - 1)];
      if (N % 4 == 0 && ldo % 4 == 0) {
        if (n < N) *reinterpret_cast<bf16x4*>(out + (int64_t)p * ldo + n) = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) out[(int64_t)p * ldo + n + r] = (bf16)v[r];
      }
    }
  }
}

// tiles: of 64 rows (ome_moe_align_tiles); A, W 16-byte aligned, lda % 8 == 0, K % 64 == 0.  runs: xcd_place
OME_API int ome_moe_gemm_stream(const void* A, int64_t lda, const int* sorted_ids, int gather_div, const void* W, const int* tiles,
                                int N, int K, int max_tiles, void* out, int64_t ldo, const void* bias, int runs, hipStream_t stream) {
  if (max_tiles <= 0) return 0;
  if (N <= 0 || K <= 0 || K % 64 || lda % 8 || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)tiles) % 16 || (uintptr_t)out % 8) return -2;
  if (max_tiles > 65535) return -3;
  const dim3 grid((N + 63) / 64, max_tiles);
  // up to two workgroups a CU: one stage more out (8 experts, 1 row: 201 -> 182 us; more of them: 398 -> 413 at 8 rows, three fit a CU)
#define ST(NST) moe_stream_kernel<64, 64, NST, 2><<<grid, 256, 0, stream>>>((const bf16*)A, lda, sorted_ids, gather_div, (const bf16*)W, \
    (const int4*)tiles, N, K, (bf16*)out, ldo, (const bf16*)bias, runs != 0)
  if ((int64_t)grid.x * max_tiles <= 512) ST(4);
  else ST(3);
#undef ST
  OME_CHECK_LAUNCH();
  return 0;
}

// bias: optional per-expert bias [E, N] added in the epilogue.  tile_m 128: the 128x128 prefill
// tile (max_m_tiles must then count 128-row tiles); otherwise the 64x64 one (any K % 32).
OME_API int ome_moe_gemm(const void* A, int64_t lda, const int* sorted_ids, int gather_div, const void* W,
                         const int* offsets, int E, int N, int K, int max_m_tiles, void* out, int64_t ldo,
                         const void* bias, int tile_m, hipStream_t stream) {
  if (max_m_tiles <= 0) return 0;
  if (K % GBK != 0 || lda % 8 != 0) return -2;
  if (max_m_tiles > 65535) return -3;
  if (tile_m == 128) {
    dim3 grid((N + 127) / 128, max_m_tiles);
    moe_gemm_v2_kernel<128, 128, 32><<<grid, 256, 0, stream>>>((const bf16*)A, lda, sorted_ids, gather_div,
                                                               (const bf16*)W, offsets, E, N, K, (bf16*)out, ldo,
                                                               (const bf16*)bias);
  } else {
    dim3 grid((N + GBN - 1) / GBN, max_m_tiles);
    moe_gemm_kernel<<<grid, 256, 0, stream>>>((const bf16*)A, lda, sorted_ids, gather_div, (const bf16*)W, offsets, E, N, K,
                                              (bf16*)out, ldo, (const bf16*)bias);
  }
  OME_CHECK_LAUNCH();
  return 0;
}

// ------------------------------------------------------------------------------------------
// combine
// ------------------------------------------------------------------------------------------
// add (optional, may alias out): out = add + scale * sum -- an always-on shared expert's output
// folded into the combine instead of a separate elementwise add
// A thread has eight columns of a token.  The experts' rows come up to eight at a time, added in their order: one after the other, each behind its
// place and weight, a row took a round trip to memory, and a workgroup took all of a token's
// columns.  us, 8 rows a token of 7168: 700 tokens 27.8 -> 18.0 (90 MB at 5.0 TB/s), 8 tokens 18.6 -> 4.8; 10 rows of 2048, 48 tokens 7.3 -> 4.8.
// PARTS: the rows as `splits` fp32 pieces `stride` floats apart, which are added first.
template <bool PARTS>
__global__ __launch_bounds__(256) void moe_combine_kernel(const void* __restrict__ Yv, const float* __restrict__ w,
                                                          const int* __restrict__ inv, int k, int H,
                                                          bf16* out, const bf16* add, float scale, int splits, int64_t stride) {
  const bf16* const Y = (const bf16*)Yv;
  const int64_t t = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= H / 8) return;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  bf16x8 a = {};
  if (add != nullptr) a = ld8(add + t * H + c * 8);
  int j = 0;
  const auto take = [&](auto count) {
    constexpr int N = decltype(count)::value;
    if constexpr (PARTS) {
      float wj[N], f[N][8];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        wj[i] = w[t * k + j + i];
        sum_parts8((const float*)Yv + (int64_t)inv[t * k + j + i] * H + c * 8, stride, splits, f[i]);
      }
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[q] += wj[i] * f[i][q];
      j += N;
      return;
    }
    bf16x8 y[N];
    float wj[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      wj[i] = w[t * k + j + i];
      y[i] = ld8(Y + (int64_t)inv[t * k + j + i] * H + c * 8);
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += wj[i] * (float)y[i][q];
    j += N;
  };
  while (k - j >= 8) take(std::integral_constant<int, 8>{});
  if (k - j >= 4) take(std::integral_constant<int, 4>{});
  if (k - j >= 2) take(std::integral_constant<int, 2>{});
  if (k - j >= 1) take(std::integral_constant<int, 1>{});
  bf16x8 o;
  if (add != nullptr) {
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = (bf16)((float)a[q] + acc[q] * scale);
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = (bf16)(acc[q] * scale);
  }
  st8(out + t * H + c * 8, o);
}

OME_API int ome_moe_combine_add(const void* Y, const float* w, const int* inv, int n_tok, int k, int H, void* out,
                                const void* add, float scale, hipStream_t stream) {
  if (n_tok <= 0) return 0;
  if (H % 8) return -2;
  moe_combine_kernel<false><<<dim3(n_tok, (H / 8 + 255) / 256), 256, 0, stream>>>(Y, w, inv, k, H, (bf16*)out, (const bf16*)add, scale, 1, 0);
  OME_CHECK_LAUNCH();
  return 0;
}

// ... of rows that ome_moe_gemm_pp left in `splits` fp32 pieces [splits][rows][H]
OME_API int ome_moe_combine_parts(const float* Y, const float* w, const int* inv, int n_tok, int k, int H, void* out,
                                  const void* add, float scale, int splits, int64_t rows, hipStream_t stream) {
  if (n_tok <= 0) return 0;
  if (H % 8 || splits < 1) return -2;
  moe_combine_kernel<true><<<dim3(n_tok, (H / 8 + 255) / 256), 256, 0, stream>>>(Y, w, inv, k, H, (bf16*)out, (const bf16*)add, scale, splits, rows * H);
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_moe_combine(const void* Y, const float* w, const int* inv, int n_tok, int k, int H, void* out,
                            float scale, hipStream_t stream) {
  return ome_moe_combine_add(Y, w, inv, n_tok, k, H, out, nullptr, scale, stream);
}

// ------------------------------------------------------------------------------------------
// FP8 block-scaled grouped GEMM (DeepSeek-V3 / Kimi-K2 `quantization: fp8` experts, SURVEY.md
// §2.9 K11): out[p, :] = dequant(A[row(p), :]) . dequant(W[e(p)])^T, A e4m3 with 1x128 group
// scales sa[row][K/128] (row = the gathered source row), W e4m3 [E][N][K] with 128x128 block scales
// sw[E][N/128][K/128].  The experts stay fp8 in HBM (half the bytes of the bf16 path, which is
// what a decode-time MoE layer is bound by).  64 x 128 tile, 4 waves (2 x 2, 32 x 64 each), one
// 128-deep K block per step = ONE v_mfma_scale_f32_16x16x128_f8f6f4 per 16 x 16 block at unit MX
// scales (2x the bf16 MFMA rate), the block's fp32 scales applied to its product with a VALU FMA.
// Operands go global -> LDS by global_load_lds (per-lane gathered source rows, lane-linear
// destination, XOR-swizzled chunks), double buffered.
// ------------------------------------------------------------------------------------------
typedef int mi32x8 __attribute__((ext_vector_type(8)));
typedef int mi32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mi32x8 mfrag32(const char* lds, int row, int c) {
  const mi32x4 lo = *reinterpret_cast<const mi32x4*>(lds + row * 128 + mswz(row, 2 * c) * 16);
  const mi32x4 hi = *reinterpret_cast<const mi32x4*>(lds + row * 128 + mswz(row, 2 * c + 1) * 16);
  return mi32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// NST LDS stages: 2 = one K block in flight during compute, waited with vmcnt(0) at the next
// step; 3 = the block two steps ahead in flight across the barrier (counted vmcnt + raw s_barrier,
// cdna_hip_programming.md "Pipelining across barriers"), at 1.5x the LDS.  All LDS is one array
// (the tile descriptor at its end): a second __shared__ object can make hipcc drain vmcnt before
// every K step's first LDS read.
template <int BMF, int BNF, int NST = 2>
__global__ __launch_bounds__(256) void moe_gemm_fp8_kernel(const uint8_t* __restrict__ A, int64_t lda,
                                                           const float* __restrict__ sa, const int* __restrict__ sorted_ids,
                                                           int gather_div, const uint8_t* __restrict__ W,
                                                           const float* __restrict__ sw, const int4* __restrict__ tiles,
                                                           int N, int K, bf16* __restrict__ out, int64_t ldo) {
  constexpr int ABYTES = BMF * 128, WBYTES = BNF * 128;
  static_assert(NST == 2 || NST == 3, "NST");
  // NST == 3 stages also carry the K block's A-row scales (4 x 256 B, one 4-byte DMA per wave):
  // an ordinary VGPR load beside the DMA makes hipcc wait vmcnt(0) and drain the ring
  constexpr int SCB = NST == 3 ? 1024 : 0, STG = ABYTES + WBYTES + SCB;
  __shared__ __attribute__((aligned(16))) char smem[NST * STG];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int4 tile = tiles[blockIdx.y];
  const int e = tile.x, m0 = tile.y, m_end = tile.z;
  if (e < 0) return;
  const bool once = __builtin_amdgcn_readfirstlane(only_tile(tiles, blockIdx.y, tile, BMF));
  const int n0 = blockIdx.x * BNF;
  const int KB = K / 128, nt = KB;
  const uint8_t* We = W + (int64_t)e * N * K;
  const float* swe = sw + ((int64_t)e * (N / 128) + n0 / 128) * KB;
  // per-lane staging sources (gathered A rows, W rows), fixed over K
  constexpr int AI = BMF / 32, WI = BNF / 32;   // wave instructions per operand per wave (8 rows each)
  const uint8_t* asrc[AI];
  const uint8_t* wsrc[WI];
#pragma unroll
  for (int j = 0; j < AI; ++j) {
    const int r = (wave * AI + j) * 8 + (lane >> 3);
    int p = m0 + r;
    p = p < m_end ? p : m_end - 1;
    const int srow = gather_div > 0 ? sorted_ids[p] / gather_div : p;
    asrc[j] = A + (int64_t)srow * lda + mswz(r, lane & 7) * 16;
  }
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int r = (wave * WI + j) * 8 + (lane >> 3);
    const int n = min(n0 + r, N - 1);
    wsrc[j] = We + (int64_t)n * K + mswz(r, lane & 7) * 16;
  }
  const float* scsrc = sa;   // NST == 3: this lane's A-row scale source (row wave*BMF/4 + lane, clamped)
  if constexpr (NST == 3) {
    const int r = wave * (BMF / 4) + min(lane, BMF / 4 - 1);
    int p = m0 + r;
    p = p < m_end ? p : m_end - 1;
    scsrc = sa + (int64_t)(gather_div > 0 ? sorted_ids[p] / gather_div : p) * (K / 128);
  }
  const auto stage_by = [&](int buf, int kt, auto policy) {
    char* la = smem + buf * STG;
    char* lw = la + ABYTES;
    if constexpr (NST == 3)
      __builtin_amdgcn_global_load_lds((moe_glb_t*)(scsrc + kt), (moe_lds_t*)(lw + WBYTES + wave * 256), 4, 0, 0);
#pragma unroll
    for (int j = 0; j < AI; ++j)
      __builtin_amdgcn_global_load_lds((moe_glb_t*)(asrc[j] + kt * 128), (moe_lds_t*)(la + (wave * AI + j) * 1024), 16,
                                       0, 0);
#pragma unroll
    for (int j = 0; j < WI; ++j)
      weights_to_lds(wsrc[j] + kt * 128, lw + (wave * WI + j) * 1024, policy);
  };
  const int wm = wave >> 1, wn = wave & 1;   // wave tile: rows [wm*BMF/2, +BMF/2), cols [wn*BNF/2, +BNF/2)
  constexpr int MJ = BMF / 32, NI = BNF / 32;
  const int fr = lane & 15, fc = lane >> 4;
  int srow[MJ];
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    int p = m0 + wm * (BMF / 2) + j * 16 + fr;
    p = p < m_end ? p : m_end - 1;
    srow[j] = gather_div > 0 ? sorted_ids[p] / gather_div : p;
  }
  f32x4 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the K block's fp32 scales are prefetched one step ahead (they ride the step's vmcnt(0) wait
  // instead of adding a dependent global-load round trip to every step)
  const float* sar[MJ];
  float san[MJ];
  float swn = 0.f;
  if constexpr (NST == 2) {
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      sar[j] = sa + (int64_t)srow[j] * KB;
      san[j] = sar[j][0];
    }
    swn = swe[0];
  }
  constexpr int NL = AI + WI + (NST == 3);   // LDS-DMA instructions per thread per K block
  const auto run = [&](const auto& stage) __attribute__((always_inline)) {
    if constexpr (NST == 2) {
      stage(0, 0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    } else {
      // blocks 0 and 1 in flight; the top of step t waits for block t with block t + 1 still out
      stage(0, 0);
      stage(1, min(1, nt - 1));
    }
    for (int t = 0; t < nt; ++t) {
      const int cur = NST == 2 ? (t & 1) : t % 3;
      if constexpr (NST == 3) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");   // block t + 1 (maybe a clamped copy) stays out
        __builtin_amdgcn_s_barrier();   // every wave's block t landed; every wave done reading block t - 1
      }
      float s[MJ];
      if constexpr (NST == 3) {
        const char* lsc = smem + cur * STG + ABYTES + WBYTES;
        const float swv = swe[t];
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          const int r = wm * (BMF / 2) + j * 16 + fr;
          s[j] = *reinterpret_cast<const float*>(lsc + (r / (BMF / 4)) * 256 + (r % (BMF / 4)) * 4) * swv;
        }
      } else {
#pragma unroll
        for (int j = 0; j < MJ; ++j) s[j] = san[j] * swn;
      }
      if constexpr (NST == 2) {
        if (t + 1 < nt) {
#pragma unroll
          for (int j = 0; j < MJ; ++j) san[j] = sar[j][t + 1];
          swn = swe[t + 1];
          stage(cur ^ 1, t + 1);
        }
      } else {
        // branch-free: the DMA of block t + 2 (into the buffer block t - 1 left) is issued every
        // step, clamped to the last block past the end, so the counted wait above stays exact
        stage((t + 2) % 3, min(t + 2, nt - 1));
      }
      const char* la = smem + cur * STG;
      const char* lw = la + ABYTES;
      mi32x8 xa[MJ];
#pragma unroll
      for (int j = 0; j < MJ; ++j) xa[j] = mfrag32(la, wm * (BMF / 2) + j * 16 + fr, fc);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const mi32x8 wf = mfrag32(lw, wn * (BNF / 2) + i * 16 + fr, fc);
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          const f32x4 p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xa[j], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0,
                                                                          127, 0, 127);
          acc[i][j] += p * s[j];
        }
      }
      if constexpr (NST == 2) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      }
    }
    if constexpr (NST == 3) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // clamped tail DMA retires before exit
  };
  if (once) run([&](int buf, int kt) { stage_by(buf, kt, ReadOnce{}); });
  else run([&](int buf, int kt) { stage_by(buf, kt, KeptWeights{}); });
  // lane (fr, fc) of block (i, j): row p = m0 + wm*BMF/2 + j*16 + fr, cols n = n0 + wn*BNF/2 + i*16 + 4fc .. +3
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int p = m0 + wm * (BMF / 2) + j * 16 + fr;
    if (p >= m_end) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = n0 + wn * (BNF / 2) + i * 16 + 4 * fc;
      if (n >= N) continue;
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (bf16)acc[i][j][r];
      *reinterpret_cast<bf16x4*>(out + (int64_t)p * ldo + n) = v;
    }
  }
}

// A [rows][K] e4m3 (gathered through sorted_ids / gather_div when gather_div > 0), sa [rows][K/128];
// W [E][N][K] e4m3, sw [E][N/128][K/128]; out [n_assign][N] bf16 in sorted order.  N % 128 == 0,
// K % 128 == 0.
// bm = 64: 64 x 128 tiles (decode: a few rows per expert, more workgroups per weight byte);
// bm = 128: 128 x 128 tiles, 64 x 64 per wave (prefill: twice the MFMAs per staged K block and the
// expert's weights read once per 128 gathered rows; 64 KB of LDS, 2 workgroups per CU).
// tiles: of bm rows (ome_moe_align_tiles), max_m_tiles of them.
OME_API int ome_moe_gemm_fp8_tile(const void* A, int64_t lda, const float* sa, const int* sorted_ids, int gather_div,
                                  const void* W, const float* sw, const int* tiles, int N, int K,
                                  int max_m_tiles, int bm, void* out, int64_t ldo, hipStream_t stream) {
  if (max_m_tiles <= 0) return 0;
  if (N % 128 || K % 128 || lda % 16 || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)tiles) % 16) return -2;
  if (max_m_tiles > 65535) return -3;
  // LDS stages (OME_MOE_FP8_NST): 3 for the 64-row tile (2 workgroups / CU, 2-5 % faster at
  // prefill sizes), 2 for the 128-row tile (3 stages = 96 KB would leave one workgroup per CU);
  // profiles/r05_fp8_moe_tiles.md
  static const int nst_env = getenv("OME_MOE_FP8_NST") ? atoi(getenv("OME_MOE_FP8_NST")) : 0;
  const int nst = nst_env ? nst_env : (bm == 64 ? 3 : 2);
#define MOE_FP8(BM, NS)                                                                                          \
  moe_gemm_fp8_kernel<BM, 128, NS><<<dim3(N / 128, max_m_tiles), 256, 0, stream>>>(                               \
      (const uint8_t*)A, lda, sa, sorted_ids, gather_div, (const uint8_t*)W, sw, (const int4*)tiles, N, K, (bf16*)out, ldo)
  if (bm == 128) {
    if (nst == 3) MOE_FP8(128, 3); else MOE_FP8(128, 2);
  } else if (bm == 64) {
    if (nst == 3) MOE_FP8(64, 3); else MOE_FP8(64, 2);
  } else {
    return -4;
  }
#undef MOE_FP8
  OME_CHECK_LAUNCH();
  return 0;
}
