// Causal prefill attention over a paged cache for four query heads to a kv head of 128 dims (Llama-3, Qwen3, Mixtral): a workgroup of two
// waves takes 32 rows (an item, or a piece of its keys), a wave those of two heads, 32 keys at a time.
//   S^T [32 keys x 32 rows] = K . Q^T    (8 products 32x32x16 a head; lane = row, eight keys of each page a lane half)
//   O^T [128 x 32 rows] += V^T . P^T     (8 products a head; V's pages hold eight keys of a dim in a row, so P^T is S^T's registers)
// A wave has its SIMD to itself (64 registers of queries, 128 of O^T, two tiles of scores), so what the matrix cores and the vector ALU do at
// once is laid out by hand: step u multiplies the scores of tile u + 1 and O^T of tile u - 1, 32 products that are independent of tile u's
// softmax, and that softmax stands beside them, a weight a product.  Every operand that comes out of LDS is used for both heads.
// O^T is rescaled where a row's largest score rose by more than 2^8, a step later than the weights (tile u - 1 is added in between).
// The first weights are of the largest score of 64 keys, as the error depends on it: with 32 it was 0.5 to 3% larger (fewer rows have a weight
// of exactly 1); with 64 it is that of the 16x16 products before, 1.76e-3 to 2.29e-3 of the result against 64 bits, to the third digit.
//
// What bounds it: a step is 32 products of 32 cycles and some 125 vector, 75 scalar, 16 LDS and 8 move instructions, which one wave issues
// at 4 cycles and more: 1850 cycles (fp8 2150: 32 conversions and 8 LDS writes).  With the chip full the products' power is the limit:
// 0.94 us a step without moves, 1140 TFLOP/s of random bf16 values (fp8's 0.80).  Time for a step of all 512 workgroups, four waves of 16x16 products
// an item -> this: bf16 1.33 -> 1.10 us, fp8 1.17 -> 1.03.  32 heads, us: 1500 rows over 7600 keys 255 -> 209 (fp8 223 -> 205), 8000 rows
// 605 -> 511 (575 -> 520), 2 x 2048 rows 94 -> 81 (94 -> 84), 4 x 500 over 900 keys 40 -> 35.5, 32 x 64 rows 13.8 -> 12.4, 8 x 256 and 300 rows
// the same.  What it does not gain: moves of 64 rows' tiles would be shared by twice the waves, but items of 32 rows fill the chip better.
#include "common.h"
#include "mma32.h"
#include "prefill_pair.h"

#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void mma_new(f32x16& c, bf16x8 a, bf16x8 b) {   // c = a b
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b) : "memory");
#endif
}
// The last products of two chains, which others read afterwards, and what fills the wait for them: two products of O^T and four exponentials.
// (In one block, as the compiler may move a result elsewhere before a wait that it sees apart from the product.)
__device__ __forceinline__ void mma_turn(f32x16& s0, f32x16& s1, bf16x8 k, bf16x8 q0, bf16x8 q1, f32x16& o0, f32x16& o1, bf16x8 v, bf16x8 p0, bf16x8 p1,
                                         float& e0, float& e1, float& e2, float& e3) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "v_mfma_f32_32x32x16_bf16 %0, %8, %9, %0\n\tv_exp_f32 %4, %4\n\t"
      "v_mfma_f32_32x32x16_bf16 %1, %8, %10, %1\n\tv_exp_f32 %5, %5\n\t"
      "v_mfma_f32_32x32x16_bf16 %2, %11, %12, %2\n\tv_exp_f32 %6, %6\n\t"
      "v_mfma_f32_32x32x16_bf16 %3, %11, %13, %3\n\tv_exp_f32 %7, %7\n\ts_nop 3"
      : "+v"(s0), "+v"(s1), "+a"(o0), "+a"(o1), "+v"(e0), "+v"(e1), "+v"(e2), "+v"(e3)
      : "v"(k), "v"(q0), "v"(q1), "v"(v), "v"(p0), "v"(p1)
      : "memory");
#endif
}
__device__ __forceinline__ void mma_last(f32x16& c, bf16x8 a, bf16x8 b) {   // c += a b, which others may read
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\t" MMA_WAIT : "+v"(c) : "v"(a), "v"(b) : "memory");
#endif
}

// A wave's two moves of 1 KiB to LDS (buffer_to_lds), the second 2048 bytes behind the first there and from `off1` + 2048
__device__ __forceinline__ void two_to_lds(const void* base, uint32_t bytes, uint32_t off0, uint32_t off1, uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint64_t b = (uint64_t)base;
  const u32x4 rs = {(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, bytes, 0x00020000u};
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\tbuffer_load_dwordx4 %2, %3, 0 offen offset:2048 lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off0), "v"(off1), "s"(rs)
               : "m0", "memory");
#endif
}

__device__ __forceinline__ void mma_acc_last(f32x16& c, bf16x8 a, bf16x8 b) {   // c += a b, the last of all
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\t" MMA_WAIT : "+a"(c) : "v"(a), "v"(b) : "memory");
#endif
}

// Keeps what computes x on this side of the next product: the compiler would sink it past them all to its use.
template <typename T>
__device__ __forceinline__ void here(T& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(x));
#endif
}

// (IEEE's maximum, one instruction of three operands: fmaxf would canonicalise each that comes out of an asm.  A NaN among a row's scores is
// one among its weights.)
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float max3(float a, float b, float c) { return max2(max2(a, b), c); }

// 16 elements of an fp8 cache -> half `HALF` of them, pair by pair
template <int F>
__device__ __forceinline__ bf16x2 fp8_pair(uint32_t w, bool hi) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (F == KV_E4M3) return hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, true) : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, false);
  else return hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.f, true) : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.f, false);
#else
  return bf16x2{};
#endif
}

#define OME_NEG_INF (-__builtin_inff())
constexpr int D = 128, P = 16, KT = 32;             // head dim, page, keys of a tile
constexpr int K_IMG = KT * D * 2, K_RING = 4, V_RING = 5;   // bytes of a tile's image of K (and of V); images

constexpr int LDO = D + 8;   // padded row of the output on its way out
static_assert(4 * 32 * LDO * 2 <= (K_RING + V_RING) * K_IMG, "it fits the images");

// Piece x of key row r of a K image lies at x ^ key_swz(r), half x of dim d of a V image at x ^ dim_swz(d): eight lanes read all banks.
__device__ __forceinline__ int key_swz(int r) { return (r & 3) | (r >> 1 & 4); }
__device__ __forceinline__ int dim_swz(int d) { return d >> 2 & 1; }

template <int F, int SPLIT>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_pair_kernel(PairArgs a) {
  constexpr int EB = F == KV_BF16 ? 2 : 1;   // bytes of a cache element
  __shared__ __attribute__((aligned(16))) char sm[(K_RING + V_RING) * K_IMG];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sm;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 31, hf = lane >> 5;
  const int kvh = blockIdx.x % a.Hkv;
  const int head = kvh * 4 + 2 * wave;   // and the next
  int e0 = blockIdx.x / a.Hkv, e1 = e0 + 1;
  const int4* list = reinterpret_cast<const int4*>(a.items);
  if constexpr (SPLIT == 2) {   // a workgroup's run of pieces, behind the pieces
    const int4 run = list[a.listed + e0];
    e0 = __builtin_amdgcn_readfirstlane(run.x), e1 = __builtin_amdgcn_readfirstlane(run.y);
  }
  // operands in their images
  uint32_t kofs[4], vofs;
  const int key = (n & 19) | (n & 4) << 1 | (n & 8) >> 1;   // slot n of a tile: S^T's rows come out as P^T's operand takes them
#pragma unroll
  for (int e = 0; e < 4; ++e) kofs[e] = key * 256 + ((2 * e + hf) ^ key_swz(key)) * 16;
  vofs = n * 32 + (hf ^ dim_swz(n)) * 16;
  for (int entry = e0; entry < e1; ++entry) {
    if (SPLIT == 2 && entry > e0) __syncthreads();   // the piece before is done with the images
    int s, r0, c_lo = 0, c_hi = 0x7fffffff, part = -1;
    if constexpr (SPLIT > 0) {
      const int4 it = list[entry];
      s = it.x, r0 = it.y, c_lo = it.z, part = it.w;
      if (a.listed > 0) {   // up to the item's next piece
        if (entry + 1 < a.listed && part >= 0) {
          const int4 nx = list[entry + 1];
          if (nx.x == s && nx.y == r0) c_hi = nx.z;
        }
      } else {
        c_hi = c_lo + a.chunk;
      }
    } else {
      const int2 it = reinterpret_cast<const int2*>(a.items)[e0];
      s = it.x, r0 = it.y;
    }
    s = __builtin_amdgcn_readfirstlane(s), r0 = __builtin_amdgcn_readfirstlane(r0);
    c_lo = __builtin_amdgcn_readfirstlane(c_lo), c_hi = __builtin_amdgcn_readfirstlane(c_hi), part = __builtin_amdgcn_readfirstlane(part);
    const int q0 = __builtin_amdgcn_readfirstlane(a.cu_q[s]), q_len = __builtin_amdgcn_readfirstlane(a.cu_q[s + 1]) - q0;
    const int kv_len = __builtin_amdgcn_readfirstlane(a.kv_lens[s]), prefix = kv_len - q_len;
    const int row = r0 + n;
    const int kv_end = min(min(kv_len, prefix + min(r0 + 32, q_len)), c_hi);
    const int begin = c_lo / KT, tiles = max((kv_end + KT - 1) / KT - begin, 0);   // (pieces start at whole tiles)
    const int* bt = a.block_tables + (int64_t)s * a.bt_stride;
    const int n_pages = (kv_len + P - 1) / P;
    const uint32_t page_bytes = a.Hkv * P * D * EB;
    const char* kc = reinterpret_cast<const char*>(a.k_cache) + (int64_t)kvh * P * D * EB;
    const char* vc = reinterpret_cast<const char*>(a.v_cache) + (int64_t)kvh * P * D * EB;

    bf16x8 qf[2][8];
    // pages of the 32 tiles from `pg0` on, one a lane
    int pages = 0, pg0 = 0;
    auto look = [&](int tile) __attribute__((always_inline)) {
      const int p = 2 * (begin + tile) + lane;
#if defined(__HIP_DEVICE_COMPILE__)   // (waited for here: the compiler would wait before every use, and for the moves as well)
      asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=&v"(pages) : "v"(bt + min(p, n_pages - 1)) : "memory");
#endif
      pg0 = tile;
    };
    // the tile of K on its way, and of V one tile behind: offsets of their pages, images
    uint64_t kpA = 0, kpB = 0, vpA = 0, vpB = 0;
    int k_at = 0, v_at = 0;
    uint32_t k_in = 0, v_in = 0;   // bytes of a page of theirs: none past the end
    auto aim = [&](int tile) __attribute__((always_inline)) {   // K of `tile`, V of the one before
      vpA = kpA, vpB = kpB, v_in = k_in;
      k_in = tile < tiles ? P * D * 2 : 0;
      if (tile - pg0 == 32 && tile < tiles) look(tile);
      const int at = 2 * (min(tile, tiles - 1) - pg0);   // (past the end: fp8 reads the last tile again)
      kpA = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(pages, at & 63) * page_bytes;
      kpB = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(pages, (at + 1) & 63) * page_bytes;
      asm("" : "+s"(kpA), "+s"(kpB));   // (in scalar registers)
    };
    // bf16: four pairs of moves of 1 KiB, j: K of pages A and B, V of pages A and B; the wave's half of a page, rows (dims) in two runs
    uint32_t koff[2], voff[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int part4 = 2 * x + wave, r = 4 * part4 + (lane >> 4);
      koff[x] = r * 256 + ((lane & 15) ^ key_swz(r)) * 16 - 2048 * x;
      voff[x] = 1024 * part4 + (lane >> 1) * 32 + ((lane & 1) ^ dim_swz(lane >> 1)) * 16 - 2048 * x;
    }
    auto dma = [&](int j) __attribute__((always_inline)) {
      if constexpr (F == KV_BF16) {
        const bool isv = j >= 2;
        const char* base = (isv ? vc : kc) + (isv ? (j & 1 ? vpB : vpA) : (j & 1 ? kpB : kpA));
        two_to_lds(base, __builtin_amdgcn_readfirstlane(isv ? v_in : k_in), isv ? voff[0] : koff[0], isv ? voff[1] : koff[1],
                   lds0 + (isv ? K_RING + v_at : k_at) * K_IMG + (j & 1) * 4096 + wave * 1024);
      }
    };
    auto advance = [&]() __attribute__((always_inline)) {
      k_at = k_at + 1 == K_RING ? 0 : k_at + 1;
      v_at = v_at + 1 == V_RING ? 0 : v_at + 1;
    };
    // fp8: 16 bytes a thread of each page of K (row tid / 8, piece tid % 8) and of V (dim tid), converted on their way
    uint4 raw[4];
    bf16x8 cv;
    uint32_t kw[2], vw[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int r = tid >> 3;   // (key_swz of r + 16 is that of r)
      kw[x] = r * 256 + ((2 * (tid & 7) + x) ^ key_swz(r)) * 16;
      vw[x] = K_RING * K_IMG + tid * 32 + (x ^ dim_swz(tid)) * 16;
    }
    auto fetch = [&](uint4 (&raw)[4], int j) __attribute__((always_inline)) {
      if constexpr (F != KV_BF16) {
        const char* base = j < 2 ? kc + (j & 1 ? kpB : kpA) : vc + (j & 1 ? vpB : vpA);
        raw[j] = *reinterpret_cast<const uint4*>(base + tid * 16);
      }
    };
    auto convert = [&](const uint4 (&raw)[4], int unit, int part) __attribute__((always_inline)) {   // unit / 2: raw piece, unit & 1: its half; in three parts
      if constexpr (F != KV_BF16) {
        const int j = unit >> 1;
        if (part < 2) {
          const uint32_t w = unit & 1 ? (part ? raw[j].w : raw[j].z) : (part ? raw[j].y : raw[j].x);
          const bf16x2 lo = fp8_pair<F>(w, false), hi = fp8_pair<F>(w, true);
          cv[4 * part] = lo[0], cv[4 * part + 1] = lo[1], cv[4 * part + 2] = hi[0], cv[4 * part + 3] = hi[1];
        } else {
          const uint32_t to = j < 2 ? kw[unit & 1] + k_at * K_IMG : vw[unit & 1] + v_at * K_IMG;
          *reinterpret_cast<bf16x8*>(sm + to + (j & 1) * 4096) = cv;
        }
      }
    };

    auto kfrag = [&](int img, int ks) __attribute__((always_inline)) { return *reinterpret_cast<const bf16x8*>(sm + (kofs[ks & 3] + img * K_IMG) + (ks >> 2) * 128); };
    auto vfrag = [&](int img, int i) __attribute__((always_inline)) {   // i: page, then 32 dims
      return *reinterpret_cast<const bf16x8*>(sm + (vofs + (K_RING + img) * K_IMG) + (i >> 2) * 4096 + (i & 3) * 1024);
    };
    auto landed = [&]() __attribute__((always_inline)) {   // (fp8: at least one read follows a step's last write)
      if constexpr (F == KV_BF16) asm volatile("s_waitcnt vmcnt(12)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt lgkmcnt(1)\n\ts_barrier" ::: "memory");
    };

    f32x16 o[2][4];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[rb][v][i] = 0.f;
    float m[2] = {OME_NEG_INF, OME_NEG_INF}, nm[2] = {0.f, 0.f}, ls[2] = {0.f, 0.f}, back[2] = {1.f, 1.f};
    int pend = 0;
    f32x16 sA[2], sB[2];
    bf16x8 pA[2][2], pB[2][2], fr[4];
    float mx[2];
    const float mul = a.mul;

    auto rescale = [&]() __attribute__((always_inline)) {   // O^T by what the maximum rose a tile ago
      asm volatile(MMA_WAIT ::: "memory");   // (without O^T as an operand: the compiler would copy it ahead of the wait, two slots behind a product)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float x = o[rb][v][i];
#if defined(__HIP_DEVICE_COMPILE__)
            float y;
            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1" : "+a"(x), "=&v"(y) : "v"(back[rb]));
#endif
            o[rb][v][i] = x;
          }
      asm volatile("s_nop 7" ::: "memory");
    };
    auto whole_row = [&](int rb) __attribute__((always_inline)) {   // a lane has half of its row's keys
      auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx[rb]), __float_as_uint(mx[rb]), false, false);
      mx[rb] = max2(__uint_as_float(w[0]), __uint_as_float(w[1])) * mul;
      here(mx[rb]);
    };
    auto rise = [&](auto once) __attribute__((always_inline)) {   // (once: there is nothing to rescale yet)   // of the tile whose rows' maxima are in mx
      const uint64_t rows = __ballot(mx[0] > m[0] + 8.f || mx[1] > m[1] + 8.f);
      const int grow = __builtin_amdgcn_readfirstlane((uint32_t)rows | (uint32_t)(rows >> 32));
      if (pend | grow) {
        asm volatile("" ::: "memory");
        if constexpr (!decltype(once)::value)
          if (pend) rescale();
        pend = grow;
        if (grow) {
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            const float m_new = fmaxf(m[rb], mx[rb]), m_use = m_new == OME_NEG_INF ? 0.f : m_new;
            back[rb] = __builtin_amdgcn_exp2f(m[rb] - m_use);
            ls[rb] *= back[rb];
            m[rb] = m_new;
            nm[rb] = -m_use;
          }
        }
      }
    };
    auto top = [&](const f32x16 (&x)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        mx[rb] = OME_NEG_INF;
#pragma unroll
        for (int i = 0; i < 16; i += 2) mx[rb] = max3(mx[rb], x[rb][i], x[rb][i + 1]);
        whole_row(rb);
      }
    };
    auto mask = [&](f32x16 (&x)[2], int tile) __attribute__((always_inline)) {
      const int base = (begin + tile) * KT;
      if (base + KT > min(prefix + r0 + 1, kv_end)) {
        asm volatile("" ::: "memory");
        const int last = min(prefix + row, kv_end - 1) - base - 8 * hf;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int i = 0; i < 16; ++i) x[rb][i] = 16 * (i >> 3) + (i & 7) > last ? OME_NEG_INF : x[rb][i];
      }
    };
    auto score = [&](f32x16 (&to)[2], int img, int tile, auto&& beside) __attribute__((always_inline)) {   // of the whole tile, with its mask
      bf16x8 k[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) k[ks] = kfrag(img, ks);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          if (ks == 0) mma_new(to[rb], k[0], qf[rb][0]);
          else if (ks < 7) mma_add(to[rb], k[ks & 3], qf[rb][ks]);
          else mma_last(to[rb], k[3], qf[rb][ks]);
          if (rb == 1 && ks < 4) k[ks] = kfrag(img, ks + 4);
          beside(2 * ks + rb);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      mask(to, tile);
    };
    auto ready = [&](bf16x8 (&p)[2][2]) __attribute__((always_inline)) {   // written by the vector ALU just now, or moved
#if defined(__HIP_DEVICE_COMPILE__)
      asm volatile("s_nop 3"
                   : "+v"(p[0][0]), "+v"(p[0][1]), "+v"(p[1][0]), "+v"(p[1][1]), "+a"(o[0][0]), "+a"(o[0][1]), "+a"(o[0][2]), "+a"(o[0][3]), "+a"(o[1][0]),
                     "+a"(o[1][1]), "+a"(o[1][2]), "+a"(o[1][3])::"memory");
#endif
    };
    auto weighted = [&](bf16x8 (&p)[2][2], int img) __attribute__((always_inline)) {   // O^T += V^T P^T
      bf16x8 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = vfrag(img, i);
      ready(p);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          if (i == 7 && rb == 1) mma_acc_last(o[rb][3], v[3], p[rb][1]);   // (others read O^T from here on)
          else mma_acc(o[rb][i & 3], v[i & 3], p[rb][i >> 2]);
        }
        if (i < 4) v[i] = vfrag(img, i + 4);
      }
    };

    int kn = 0, vn = 0;   // image of K of tile u + 1, of V of tile u - 1
    auto next_k = [&](int x) { return x + 1 == K_RING ? 0 : x + 1; };
    auto next_v = [&](int x) { return x + 1 == V_RING ? 0 : x + 1; };
    // Step u: the scores of tile u + 1 (those between the first and the last step), O^T of tile u - 1 (those and the last), and beside their products the
    // weights of tile u and the maxima of tile u + 1.  MASKED: tile u + 1 may be one that not all rows see.
    enum { WHOLE, MASKED, FIRST, LAST };
    auto step = [&](int u, f32x16 (&x)[2], f32x16 (&y)[2], bf16x8 (&po)[2][2], bf16x8 (&pn)[2][2], auto which) __attribute__((always_inline)) {
      constexpr int KIND = decltype(which)::value;
      const int k2 = next_k(kn);
      float w[32];
      uint32_t pk[16];
      const auto arg = [&](int i) __attribute__((always_inline)) {
        w[i] = __builtin_fmaf(x[i >> 4][i & 15], mul, nm[i >> 4]);
        here(w[i]);
      };
      const auto weight = [&](int i) __attribute__((always_inline)) {
        w[i] = __builtin_amdgcn_exp2f(w[i]);
        here(w[i]);
      };
      const auto sum = [&](int i) __attribute__((always_inline)) {
        ls[i >> 4] += w[i];
        here(ls[i >> 4]);
        if (i & 1) {
          pk[i >> 1] = __builtin_bit_cast(uint32_t, bf16x2{(bf16)w[i - 1], (bf16)w[i]});
          here(pk[i >> 1]);
        }
        if ((i & 7) == 7) pn[i >> 4][i >> 3 & 1] = __builtin_bit_cast(bf16x8, u32x4{pk[i / 8 * 4], pk[i / 8 * 4 + 1], pk[i / 8 * 4 + 2], pk[i / 8 * 4 + 3]});
      };
      const auto two = [&](int i) __attribute__((always_inline)) {   // weights 2 i and 2 i + 1, a product behind
        if (i > 0) sum(2 * i - 2), sum(2 * i - 1);
        if (i < 16) {
          arg(2 * i), arg(2 * i + 1);
          weight(2 * i), weight(2 * i + 1);
        }
      };
      const auto stage = [&](int i) __attribute__((always_inline)) {   // 28 pieces of what brings in the next tiles
        if constexpr (F == KV_BF16) {
          if (i < 16 && i % 4 == 0) dma(i / 4);
        } else {
          const int at = i % 14, half = i / 14;   // units of three pieces, four in each half
          if (at < 12) convert(raw, at / 3 + 4 * half, at % 3);
          if (at == 6 || at == 12) fetch(raw, (at == 6 ? 0 : 1) + 2 * half);   // (read two thirds of a step later)
        }
      };
      if constexpr (KIND != LAST) aim(u + 4);
      if constexpr (KIND == LAST) {
        if (tiles > 1) {
#pragma unroll
          for (int e = 0; e < 4; ++e) fr[e] = vfrag(vn, e);
          ready(po);
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
              mma_acc(o[rb][e & 3], fr[e & 3], po[rb][e >> 2]);
              if (rb == 1 && e < 4) fr[e] = vfrag(vn, e + 4);
              two(2 * e + rb);
              __builtin_amdgcn_sched_barrier(0);
            }
          vn = next_v(vn);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) two(i);
        }
        two(16);
        if (__builtin_amdgcn_readfirstlane(pend)) rescale();
        return;
      }
      if constexpr (KIND == FIRST) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          two(i);
          if (i < 14) stage(2 * i), stage(2 * i + 1);
          if (i >= 12) fr[i - 12] = kfrag(k2, i - 12);
          __builtin_amdgcn_sched_barrier(0);
        }
        two(16);
      } else {
        const auto beside = [&](int i) __attribute__((always_inline)) {   // products 0..13 and 18..31
          weight(i);
          if (i == 13) {
#pragma unroll
            for (int e = 14; e < 19; ++e) arg(e);
          } else if (i + 1 < 32) {
            arg(i + 1);
          }
          if (i < 14) {
            if (i > 0) sum(i - 1);
          } else if (i < 22) {
            sum(13 + 2 * (i - 18));
            sum(14 + 2 * (i - 18));
          } else {
            sum(i - 1);
          }
          if (i >= 18 && i < 30) {   // the maxima, in pairs
#pragma unroll
            for (int e = (i - 18) * 16 / 12; e < (i - 17) * 16 / 12; ++e) {
              const int rb = e >> 3, k = 2 * (e & 7);
              mx[rb] = k == 0 ? max2(y[rb][0], y[rb][1]) : max3(mx[rb], y[rb][k], y[rb][k + 1]);
              here(mx[rb]);
            }
          }
          if (i == 26) whole_row(0);
          if (i == 30) whole_row(1);
          stage(i < 14 ? i : i - 4);
        };
        arg(0);
#pragma unroll
        for (int e = 0; e < 7; ++e)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            if (e == 0) mma_new(y[rb], fr[0], qf[rb][0]);
            else mma_add(y[rb], fr[e & 3], qf[rb][e]);
            if (rb == 1) fr[e & 3] = e < 4 ? kfrag(kn, e + 4) : vfrag(vn, e - 4);
            beside(2 * e + rb);
            __builtin_amdgcn_sched_barrier(0);
          }
        mma_turn(y[0], y[1], fr[3], qf[0][7], qf[1][7], o[0][0], o[1][0], fr[0], po[0][0], po[1][0], w[14], w[15], w[16], w[17]);
        fr[3] = vfrag(vn, 3);
        fr[0] = vfrag(vn, 4);
        if constexpr (KIND == MASKED) mask(y, u + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 1; e < 8; ++e)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            mma_acc(o[rb][e & 3], fr[e & 3], po[rb][e >> 2]);
            if (rb == 1) fr[e & 3] = e < 4 ? vfrag(vn, e + 4) : kfrag(k2, e & 3);
            beside(16 + 2 * e + rb);
            __builtin_amdgcn_sched_barrier(0);
          }
        sum(31);
        vn = next_v(vn);
      }
      kn = k2;
      advance();
      if constexpr (KIND != FIRST) rise(std::false_type{});
      landed();
    };

    if (tiles > 0) {
      {   // queries and pages (by asm: the compiler would wait for them at their first use, and for the moves as well)
        const bf16* qa = a.q + (int64_t)(q0 + min(row, q_len - 1)) * a.q_stride + (int64_t)head * D + 8 * hf;
        const int* pa = bt + min(2 * begin + lane, n_pages - 1);
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile(
            "global_load_dword %16, %18, off\n\t"
            "global_load_dwordx4 %0, %17, off\n\tglobal_load_dwordx4 %1, %17, off offset:32\n\t"
            "global_load_dwordx4 %2, %17, off offset:64\n\tglobal_load_dwordx4 %3, %17, off offset:96\n\t"
            "global_load_dwordx4 %4, %17, off offset:128\n\tglobal_load_dwordx4 %5, %17, off offset:160\n\t"
            "global_load_dwordx4 %6, %17, off offset:192\n\tglobal_load_dwordx4 %7, %17, off offset:224\n\t"
            "global_load_dwordx4 %8, %17, off offset:256\n\tglobal_load_dwordx4 %9, %17, off offset:288\n\t"
            "global_load_dwordx4 %10, %17, off offset:320\n\tglobal_load_dwordx4 %11, %17, off offset:352\n\t"
            "global_load_dwordx4 %12, %17, off offset:384\n\tglobal_load_dwordx4 %13, %17, off offset:416\n\t"
            "global_load_dwordx4 %14, %17, off offset:448\n\tglobal_load_dwordx4 %15, %17, off offset:480\n\ts_waitcnt vmcnt(0)"
            : "=&v"(qf[0][0]), "=&v"(qf[0][1]), "=&v"(qf[0][2]), "=&v"(qf[0][3]), "=&v"(qf[0][4]), "=&v"(qf[0][5]), "=&v"(qf[0][6]), "=&v"(qf[0][7]),
              "=&v"(qf[1][0]), "=&v"(qf[1][1]), "=&v"(qf[1][2]), "=&v"(qf[1][3]), "=&v"(qf[1][4]), "=&v"(qf[1][5]), "=&v"(qf[1][6]), "=&v"(qf[1][7]),
              "=&v"(pages)
            : "v"(qa), "v"(pa)
            : "memory");
#endif
      }
      uint4 first[3][4];
      // K of tiles 0..3, V of tiles 0..2 (fp8: the last of each stay on their way)
      if constexpr (F == KV_BF16) {
#pragma unroll 1
        for (int t = 0; t < 4; ++t) {
          aim(t);
          k_at = t, v_at = t - 1;
          dma(0), dma(1);
          if (t > 0) dma(2), dma(3);
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          aim(t);
#pragma unroll
          for (int j = 0; j < (t > 0 ? 4 : 2); ++j) fetch(t < 3 ? first[t] : raw, j);
        }
#pragma unroll
        for (int x = 0; x < 8; ++x)
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            k_at = x / 4;
            convert(first[x / 4], x % 4, p);
          }
      }
      if constexpr (F == KV_BF16) asm volatile("s_waitcnt vmcnt(20)\n\ts_barrier" ::: "memory");   // K of tiles 0 and 1
      else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      score(sA, 0, 0, [&](int i) __attribute__((always_inline)) {
        if constexpr (F != KV_BF16) {   // the other conversions beside it: V of tile 0, K of tile 2, V of tile 1
          const int unit = i < 4 ? 4 + i : i < 8 ? i - 4 : i - 4;
          k_at = 2, v_at = i < 4 ? 0 : 1;
          if (i < 12)
#pragma unroll
            for (int p = 0; p < 3; ++p) convert(first[i < 4 ? 1 : 2], unit, p);
        }
      });
      top(sA);
      if (tiles > 1) {   // the first weights are of the largest score of 64 keys: the largest is exactly 1 then
        const float m0 = mx[0], m1 = mx[1];
        score(sB, 1, 1, [](int) {});
        top(sB);
        mx[0] = max2(mx[0], m0), mx[1] = max2(mx[1], m1);
      }
      rise(std::true_type{});
      pend = 0;
      if constexpr (F != KV_BF16) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      landed();   // (and step 0 moves a tile to the image of K just read)
      // where step 0 writes: bf16 K of tile 4 and V of tile 3, fp8 of tiles 3 and 2
      k_at = F == KV_BF16 ? 0 : 3, v_at = F == KV_BF16 ? 3 : 2;
      kn = 1, vn = 0;
      int u = 0;
      if (tiles > 1) {
        step(0, sA, sB, pB, pA, std::integral_constant<int, FIRST>{});
        sA[0] = sB[0], sA[1] = sB[1];
        u = 1;
        const int fast = min(min(prefix + r0 + 1, kv_end) / KT - begin, tiles) - 1;   // steps whose next tile all rows see
        for (; u + 1 < fast; u += 2) {
          step(u, sA, sB, pA, pB, std::integral_constant<int, WHOLE>{});
          step(u + 1, sB, sA, pB, pA, std::integral_constant<int, WHOLE>{});
        }
#pragma unroll 1
        for (; u + 1 < tiles; ++u) {
          step(u, sA, sB, pA, pB, std::integral_constant<int, MASKED>{});
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            sA[rb] = sB[rb];
            pA[rb][0] = pB[rb][0], pA[rb][1] = pB[rb][1];
          }
        }
      }
      step(u, sA, sB, pA, pB, std::integral_constant<int, LAST>{});
      weighted(pB, vn);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");   // (the images are done with)

#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(ls[rb]), __float_as_uint(ls[rb]), false, false);
      ls[rb] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
      const bool split = SPLIT > 0 && part >= 0;
      const float lt = a.sinks ? ls[rb] + __builtin_amdgcn_exp2f(a.sinks[head + rb] * 1.4426950408889634f - m[rb]) : ls[rb];
      const float f = split ? 1.f : lt > 0.f ? a.v_scale / lt : 0.f;
      f32x4 x[4][4];
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int i = 0; i < 16; ++i) x[v][i / 4][i % 4] = o[rb][v][i] * f;
      if (split) {   // unnormalised, in the lanes' own order: dim 32 v + 8 i + 4 hf + e of row n
        const int64_t pw = ((int64_t)part * a.Hkv + kvh) * 4 + 2 * wave + rb;
        float* po = a.part_o + pw * 32 * D + 4 * lane;
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(po + (4 * v + i) * 256) = x[v][i];
        if (hf == 0) *reinterpret_cast<float2*>(a.part_ml + (pw * 32 + n) * 2) = make_float2(m[rb], ls[rb]);
      } else {   // through LDS, so that rows leave whole
        bf16* so = reinterpret_cast<bf16*>(sm) + (2 * wave + rb) * 32 * LDO;
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            *reinterpret_cast<bf16x4*>(so + n * LDO + 32 * v + 8 * i + 4 * hf) = bf16x4{(bf16)x[v][i][0], (bf16)x[v][i][1], (bf16)x[v][i][2], (bf16)x[v][i][3]};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (a wave's own rows)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = 4 * i + (lane >> 4);
          if (r0 + r < q_len)
            st8(a.out + (int64_t)(q0 + r0 + r) * a.out_stride + (int64_t)(head + rb) * D + 8 * (lane & 15), ld8(so + r * LDO + 8 * (lane & 15)));
        }
      }
    }
  }
}

template <int F>
void launch(const PairArgs& a, int split, int grid, hipStream_t stream) {
  if (split == 2) prefill_pair_kernel<F, 2><<<grid, 128, 0, stream>>>(a);
  else if (split == 1) prefill_pair_kernel<F, 1><<<grid, 128, 0, stream>>>(a);
  else prefill_pair_kernel<F, 0><<<grid, 128, 0, stream>>>(a);
}

}  // namespace

void ome_prefill_pair(const PairArgs& a, int kv_fmt, int split, int grid, hipStream_t stream) {
  if (kv_fmt == KV_BF16) launch<KV_BF16>(a, split, grid, stream);
  else if (kv_fmt == KV_E4M3) launch<KV_E4M3>(a, split, grid, stream);
  else launch<KV_E5M2>(a, split, grid, stream);
}
