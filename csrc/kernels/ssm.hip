// Mamba-2 (selective state space) kernels for hybrid models (NemotronH; reference catalog
// ``NemotronHForCausalLM`` runtimes), CDNA4 / gfx950.
//
//   ome_ssm_conv1d       : causal depthwise conv (K <= 32 taps) + SiLU over a varlen batch of
//                          sequences, continuing from / updating each sequence's conv state
//   ome_dyn_conv1d       : the same with per-row (input-generated) taps (Jet-Nemotron JetBlock)
//   ome_ssm_scan         : the selective scan  h <- exp(dt*A) h + dt * B x,  y = C.h + D x
//                          (dt = softplus(dt + dt_bias) clamped below), recurrent over the rows of
//                          each sequence, state in fp32 per (slot, head, p, n)
//   ome_gated_rmsnorm    : out = w * groupRMSNorm(y * silu(z))  (norm_first: w[:group] * groupRMSNorm(y) * silu(z),
//                          or * sigmoid(z))
//
// Sequences are described by cu[S+1] (row ranges), slot[S] (state row) and reset[S] (1 = start
// from zero state: a sequence's first prefill chunk).  Decode is the S = batch, one-row case, so
// the same launches are captured in the decode HIP graph.
//
// Scan layout: one 256-thread workgroup per (head, sequence); the head's P x N state is split so
// that TPP = 256 / P consecutive lanes own one p row, NPT = N / TPP states each, held in VGPRs for
// the whole sequence.  Per row every lane reads its NPT B and C values straight from global (the
// TPP lanes of a p row read disjoint slices; the 256/TPP rows of the block read the same lines, so
// each B/C line is fetched once per wave through the vector cache) -- no LDS and no barrier in the
// time loop; y = C.h is a TPP-lane shuffle reduction.
#include "common.h"

#include <cstdlib>

namespace {

typedef float f32v4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(__expf(x)); }
// x / (1 + e^-x): a quarter of both (so that the reciprocal of no finite denominator is subnormal), the reciprocal and the quotient
// with a Newton step each: eight instructions for the compiler's division's eleven, and the same bf16 for every bf16 x
__device__ __forceinline__ float silu_f(float x) {
  const float n = 0.25f * x, d = __builtin_fmaf(__expf(-x), 0.25f, 0.25f), r0 = __builtin_amdgcn_rcpf(d);
  const float r = __builtin_fmaf(__builtin_fmaf(-d, r0, 1.f), r0, r0), q = n * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, n), r, q), d, n);   // (infinities and NaN)
}

// Causal depthwise conv + SiLU, K <= 6 taps.  Not recurrent, so rows are parallel: a wave owns 64 * V
// neighbouring channels (V = 8: 16-byte row pieces) of a tile of CT rows and slides a register window over
// them, CR rows computed while the next CR are on their way.  Tiles belong to sequences: sequence s owns tile ids cu[s] / CT + s and
// up (never overlapping, below T / CT + S).  Only a sequence's first tile touches the state (K - 1 <= CT): it
// reads the old tail before its rows and writes the new one, from the sequence's last rows or, where it is
// shorter than K - 1, from the old tail shifted; no other tile races with it.  `by_seq` (decode steps, no more
// rows than sequences): wave id = sequence, all its rows, without the search.  `out` must not overlap `x`.
// Memory-bound where rows are many, a wave's chain where they are few, so tiles are short (they read K - 1 rows again, from L2):
// 16 rows in two halves without a load ahead -> with one -> 8 rows in halves of 4 and the quotient of silu_f, us: 4000 x 8192 31 -> 34 ->
// 27.6 (4.8 TB/s), 3500 x 10240 35 -> 38 -> 29, 8000 x 2560 24.5 -> 28 -> 21, 1000 x 8192 17.9 -> 16.6 -> 10.2, 300 x 10240 11.7 -> 9.8 ->
// 7.8; 32 rows a tile 33, 43, 31, 17, 15.
constexpr int CT = 8, CR = 4;

template <int K, int V>
__global__ __launch_bounds__(256) void ssm_conv1d_kernel(const bf16* __restrict__ x, int64_t x_stride,
                                                         const bf16* __restrict__ w, const bf16* __restrict__ bias,
                                                         bf16* __restrict__ out, int64_t out_stride,
                                                         bf16* __restrict__ state, const int* __restrict__ cu,
                                                         const int* __restrict__ slot, const int* __restrict__ reset,
                                                         int S, int C, int by_seq) {
  typedef bf16 vec __attribute__((ext_vector_type(V)));
  const int lane = threadIdx.x & 63, id = blockIdx.x * 4 + (threadIdx.x >> 6);
  int s = by_seq ? id : -1;
  if (by_seq) {
    if (s >= S) return;
  } else {
    for (int b = 0; b < S; b += 64) {   // the last sequence whose first tile is not past this one
      const int i = b + lane, n = __popcll(__ballot(i < S && cu[min(i, S)] / CT + i <= id));
      s += n;
      if (n < 64) break;
    }
    if (s < 0) return;
  }
  const int r0 = cu[s], r1 = cu[s + 1], tile = by_seq ? 0 : id - (r0 / CT + s), a = r0 + tile * CT;
  const int c = (blockIdx.y * 64 + lane) * V;
  if (a >= r1 || c >= C) return;
  const int e = by_seq ? r1 : min(a + CT, r1);
  float win[K - 1][V], wt[K][V], bs[V];
#pragma unroll
  for (int t = 0; t < K; ++t) {   // taps [C, K]: K vectors hold this lane's V * K of them
    const vec v = *reinterpret_cast<const vec*>(w + (int64_t)c * K + V * t);
#pragma unroll
    for (int u = 0; u < V; ++u) wt[(V * t + u) % K][(V * t + u) / K] = (float)v[u];
  }
  {
    vec v{};
    if (bias != nullptr) v = *reinterpret_cast<const vec*>(bias + c);
#pragma unroll
    for (int u = 0; u < V; ++u) bs[u] = (float)v[u];
  }
  if (tile == 0) {
    vec* st = reinterpret_cast<vec*>(state + ((int64_t)slot[s] * C + c) * (K - 1));
    const bool fresh = reset[s] != 0;
    vec nw[K - 1];
#pragma unroll
    for (int t = 0; t < K - 1; ++t) {
      vec v{};
      if (!fresh) v = st[t];
#pragma unroll
      for (int u = 0; u < V; ++u) win[(V * t + u) % (K - 1)][(V * t + u) / (K - 1)] = (float)v[u];
    }
    const int n = r1 - r0;
#pragma unroll
    for (int t = 0; t < K - 1; ++t) {   // new tail entry t = input n - (K - 1) + t of the sequence; negative: old tail
      const int i = n - (K - 1) + t;
      vec v{};
      if (i >= 0) {
        v = *reinterpret_cast<const vec*>(x + (int64_t)(r0 + i) * x_stride + c);
      } else {
#pragma unroll
        for (int q = 0; q < K - 1; ++q)
          if (q == K - 1 + i) {
#pragma unroll
            for (int u = 0; u < V; ++u) v[u] = (bf16)win[q][u];
          }
      }
#pragma unroll
      for (int u = 0; u < V; ++u) nw[(u * (K - 1) + t) / V][(u * (K - 1) + t) % V] = v[u];
    }
#pragma unroll
    for (int t = 0; t < K - 1; ++t) st[t] = nw[t];
  } else {
#pragma unroll
    for (int t = 0; t < K - 1; ++t) {
      const vec v = *reinterpret_cast<const vec*>(x + (int64_t)(a - (K - 1) + t) * x_stride + c);
#pragma unroll
      for (int u = 0; u < V; ++u) win[t][u] = (float)v[u];
    }
  }
  vec xs[2][CR];   // rows on their way while the ones before them are computed
  const auto fetch = [&](vec (&to)[CR], int r) {
#pragma unroll
    for (int i = 0; i < CR; ++i) to[i] = *reinterpret_cast<const vec*>(x + (int64_t)min(r + i, e - 1) * x_stride + c);
  };
  const auto rows = [&](const vec (&xs)[CR], int r) {
#pragma unroll
    for (int i = 0; i < CR; ++i) {
      if (r + i >= e) break;
      vec o;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const float v = (float)xs[i][u];
        float acc = bs[u] + wt[K - 1][u] * v;
#pragma unroll
        for (int t = 0; t < K - 1; ++t) acc += wt[t][u] * win[t][u];
#pragma unroll
        for (int t = 0; t < K - 2; ++t) win[t][u] = win[t + 1][u];
        win[K - 2][u] = v;
        o[u] = (bf16)silu_f(acc);
      }
      *reinterpret_cast<vec*>(out + (int64_t)(r + i) * out_stride + c) = o;
    }
  };
  fetch(xs[0], a);
  for (int r = a; r < e; r += 2 * CR) {
    if (r + CR < e) fetch(xs[1], r + CR);
    rows(xs[0], r);
    if (r + CR >= e) break;
    if (r + 2 * CR < e) fetch(xs[0], r + 2 * CR);
    rows(xs[1], r + CR);
  }
}

// Dynamic (input-conditioned) causal depthwise conv + SiLU (Jet-Nemotron's JetBlock value path):
// every row r brings its own taps kern[r][(c / cpk) * K + j] (cpk channels share a kernel: 1 =
// per-channel, head_v_dim = per-head), tap K-1 on the current row.  Same varlen / state contract
// as ssm_conv1d_kernel.
template <int K>
__global__ __launch_bounds__(256) void dyn_conv1d_kernel(const bf16* __restrict__ x, int64_t x_stride,
                                                         const bf16* __restrict__ kern, int64_t k_stride, int cpk,
                                                         bf16* __restrict__ out, int64_t out_stride,
                                                         bf16* __restrict__ state, const int* __restrict__ cu,
                                                         const int* __restrict__ slot, const int* __restrict__ reset,
                                                         int C) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (c >= C) return;
  const int r0 = cu[s], r1 = cu[s + 1];
  if (r1 <= r0) return;
  bf16* st = state + ((int64_t)slot[s] * C + c) * (K - 1);
  float win[K - 1];
  const bool fresh = reset[s] != 0;
#pragma unroll
  for (int j = 0; j < K - 1; ++j) win[j] = fresh ? 0.f : (float)st[j];
  const int64_t kc = (int64_t)(c / cpk) * K;
  for (int r = r0; r < r1; ++r) {
    const float v = (float)x[(int64_t)r * x_stride + c];
    const bf16* kr = kern + (int64_t)r * k_stride + kc;
    float acc = (float)kr[K - 1] * v;
#pragma unroll
    for (int j = 0; j < K - 1; ++j) acc += (float)kr[j] * win[j];
#pragma unroll
    for (int j = 0; j < K - 2; ++j) win[j] = win[j + 1];
    win[K - 2] = v;
    out[(int64_t)r * out_stride + c] = (bf16)silu_f(acc);
  }
#pragma unroll
  for (int j = 0; j < K - 1; ++j) st[j] = (bf16)win[j];
}

template <int NPT, bool NT>
__global__ __launch_bounds__(256) void ssm_scan_kernel(
    const bf16* __restrict__ x, int64_t x_stride, const bf16* __restrict__ dt, int64_t dt_stride,
    const bf16* __restrict__ B, const bf16* __restrict__ Cm, int64_t bc_stride, const float* __restrict__ A,
    const float* __restrict__ D, const float* __restrict__ dt_bias, float dt_min, float* __restrict__ state,
    bf16* __restrict__ y, int64_t y_stride, const int* __restrict__ cu, const int* __restrict__ slot,
    const int* __restrict__ reset, int H, int P, int N, int G, int PB) {
  // a workgroup owns PB of the head's P rows (P / PB workgroups per head and sequence)
  const int split = P / PB;
  const int h = blockIdx.x / split, s = blockIdx.y;
  const int r0 = cu[s], r1 = cu[s + 1];
  if (r1 <= r0) return;
  const int TPP = 256 / PB;
  const int p = (blockIdx.x % split) * PB + threadIdx.x / TPP, q = threadIdx.x % TPP;
  const int n0 = q * NPT;
  const int g = h / (H / G);
  // state row: NPT contiguous fp32 per lane, a wave covers one contiguous 64*NPT*4-byte span:
  // moved with 16-B vector loads / stores (decode is bound by this state traffic)
  f32v4* st4 = reinterpret_cast<f32v4*>(state + (((int64_t)slot[s] * H + h) * P + p) * N + n0);
  float hs[NPT];
  if (reset[s] != 0) {
#pragma unroll
    for (int j = 0; j < NPT; ++j) hs[j] = 0.f;
  } else {
#pragma unroll
    for (int j = 0; j < NPT / 4; ++j) {
      const f32v4 v = NT ? __builtin_nontemporal_load(st4 + j) : st4[j];
      hs[4 * j] = v.x, hs[4 * j + 1] = v.y, hs[4 * j + 2] = v.z, hs[4 * j + 3] = v.w;
    }
  }
  const float a = A[h], d = D[h], db = dt_bias[h];
  const int64_t boff = (int64_t)g * N + n0;
  // software pipeline: the next row's dt / x / B / C are loaded while this row's FMAs run
  bf16x8 bn[NPT / 8], cn[NPT / 8];
  float dtn = 0.f, xn = 0.f;
  auto fetch = [&](int r) {
    dtn = (float)dt[(int64_t)r * dt_stride + h];
    xn = (float)x[(int64_t)r * x_stride + h * P + p];
#pragma unroll
    for (int j = 0; j < NPT / 8; ++j) {
      bn[j] = ld8(B + (int64_t)r * bc_stride + boff + 8 * j);
      cn[j] = ld8(Cm + (int64_t)r * bc_stride + boff + 8 * j);
    }
  };
  fetch(r0);
  for (int r = r0; r < r1; ++r) {
    bf16x8 bv[NPT / 8], cv[NPT / 8];
#pragma unroll
    for (int j = 0; j < NPT / 8; ++j) bv[j] = bn[j], cv[j] = cn[j];
    const float dtr = dtn, xv = xn;
    if (r + 1 < r1) fetch(r + 1);
    const float dtv = fmaxf(softplus_f(dtr + db), dt_min);
    const float dA = __expf(dtv * a);
    const float dx = dtv * xv;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < NPT / 8; ++j)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        hs[8 * j + k] = hs[8 * j + k] * dA + dx * (float)bv[j][k];
        acc += (float)cv[j][k] * hs[8 * j + k];
      }
    for (int off = 1; off < TPP; off <<= 1) acc += __shfl_xor(acc, off);
    if (q == 0) y[(int64_t)r * y_stride + h * P + p] = (bf16)(acc + d * xv);
  }
#pragma unroll
  for (int j = 0; j < NPT / 4; ++j)
  {
    const f32v4 v{hs[4 * j], hs[4 * j + 1], hs[4 * j + 2], hs[4 * j + 3]};
    if constexpr (NT) {
      __builtin_nontemporal_store(v, st4 + j);
    } else {
      st4[j] = v;
    }
  }
}

// T = float (fp32 models): no intermediate rounding; bf16: the normalised value is rounded before
// the scale, as the reference implementations of the bf16 families do.
template <typename T>
__global__ __launch_bounds__(256) void gated_rmsnorm_kernel(const T* __restrict__ y, int64_t y_stride,
                                                            const T* __restrict__ z, int64_t z_stride,
                                                            const T* __restrict__ w, T* __restrict__ out,
                                                            int64_t out_stride, int group, float eps, int mode) {
  __shared__ float red[4];
  const int norm_first = mode & 1;
  const bool exact = (mode & 2) != 0, sig = (mode & 4) != 0;   // sig: sigmoid(z) instead of silu(z) (exact, norm first)
  const int row = blockIdx.y, g0 = blockIdx.x * group;
  const T* yr = y + (int64_t)row * y_stride + g0;
  const T* zr = z + (int64_t)row * z_stride + g0;
  float ss = 0.f;
  for (int i = threadIdx.x; i < group; i += 256) {
    const float v = norm_first ? (float)yr[i] : (float)yr[i] * silu_f((float)zr[i]);
    ss += v * v;
  }
  const float tot = block_sum<256>(ss, red);
  const float rs = 1.f / sqrtf(tot / (float)group + eps);
  T* orow = out + (int64_t)row * out_stride + g0;
  for (int i = threadIdx.x; i < group; i += 256) {
    if (exact) {        // one rounding, at the store (models that keep their norms in fp32)
      const float zs = sig ? 1.f / (1.f + __expf(-(float)zr[i])) : silu_f((float)zr[i]);
      orow[i] = (T)(norm_first ? (float)yr[i] * rs * (float)w[i] * zs : (float)yr[i] * zs * rs * (float)w[g0 + i]);
    } else if (norm_first) {   // Qwen3-Next: w (per group channel) * norm(y), then * silu(z)
      const float t = (float)(T)((float)(T)((float)yr[i] * rs) * (float)w[i]);
      orow[i] = (T)(t * silu_f((float)zr[i]));
    } else {
      const float v = (float)yr[i] * silu_f((float)zr[i]) * rs;
      orow[i] = (T)((float)(T)v * (float)w[g0 + i]);  // HF: normalise, cast, then scale by w
    }
  }
}

// bf16 groups of 8 L N channels (L = 8 .. 64 lanes, N passes), every mode: a lane holds N 16-byte pieces of y and
// z, so each is read once, and a group's sum of squares stays within its L lanes (no LDS, no barrier; the block-wide
// kernel above read y twice, in 2-byte pieces, behind two barriers).  Memory-bound: 4000 x 4096 in groups of 128
// 104 -> 21 us, 3500 x 8192 in groups of 1024 116 -> 29 (42 with the gate computed once for the sum and once for the output).
template <int L, int N>
__global__ __launch_bounds__(256) void gated_rmsnorm_vec_kernel(const bf16* __restrict__ y, int64_t y_stride,
                                                                const bf16* __restrict__ z, int64_t z_stride,
                                                                const bf16* __restrict__ w, bf16* __restrict__ out,
                                                                int64_t out_stride, int64_t n, int per_row, float eps,
                                                                int mode) {
  constexpr int GROUP = 8 * L * N;
  const bool norm_first = (mode & 1) != 0, exact = (mode & 2) != 0, sig = (mode & 4) != 0;
  const int64_t id = (int64_t)blockIdx.x * (256 / L) + threadIdx.x / L;
  if (id >= n) return;   // whole groups of L lanes
  const int64_t row = id / per_row;
  const int g0 = (int)(id - row * per_row) * GROUP, l = threadIdx.x % L;
  bf16x8 yv[N], zv[N];
#pragma unroll
  for (int p = 0; p < N; ++p) {
    const int i = g0 + (l + L * p) * 8;
    yv[p] = ld8(y + row * y_stride + i);
    zv[p] = ld8(z + row * z_stride + i);
  }
  float ss = 0.f, v[N][8];   // what is normalised
#pragma unroll
  for (int p = 0; p < N; ++p)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[p][e] = norm_first ? (float)yv[p][e] : (float)yv[p][e] * silu_f((float)zv[p][e]);
      ss += v[p][e] * v[p][e];
    }
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float rs = 1.f / sqrtf(ss / (float)GROUP + eps);
#pragma unroll
  for (int p = 0; p < N; ++p) {
    const int i = (l + L * p) * 8;
    const bf16x8 wv = ld8(w + (norm_first ? i : g0 + i));
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float vv = v[p][e], zz = (float)zv[p][e], ww = (float)wv[e];
      if (norm_first) {
        if (exact) o[e] = (bf16)(vv * rs * ww * (sig ? 1.f / (1.f + __expf(-zz)) : silu_f(zz)));
        else o[e] = (bf16)((float)(bf16)((float)(bf16)(vv * rs) * ww) * silu_f(zz));
      } else {
        o[e] = (bf16)(exact ? vv * rs * ww : (float)(bf16)(vv * rs) * ww);
      }
    }
    st8(out + row * out_stride + g0 + i, o);
  }
}

// Small groups in exact mode, norm first: one wave per group, V neighbouring elements per lane and pass.
template <typename T, int V>
__global__ __launch_bounds__(256) void gated_rmsnorm_wave_kernel(const T* __restrict__ y, int64_t y_stride,
                                                                 const T* __restrict__ z, int64_t z_stride,
                                                                 const T* __restrict__ w, T* __restrict__ out,
                                                                 int64_t out_stride, int64_t n, int per_row, int group,
                                                                 float eps, int sig) {
  typedef T vec __attribute__((ext_vector_type(V)));
  const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= n) return;
  const int lane = threadIdx.x & 63, g0 = (int)(id % per_row) * group;
  const int64_t row = id / per_row;
  constexpr int NP = 8 / V;   // passes: groups of up to 512
  vec yv[NP], zv[NP];
  float ss = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = (lane + 64 * p) * V;
    if (i < group) {
      yv[p] = *reinterpret_cast<const vec*>(y + row * y_stride + g0 + i);
      zv[p] = *reinterpret_cast<const vec*>(z + row * z_stride + g0 + i);
#pragma unroll
      for (int e = 0; e < V; ++e) ss += (float)yv[p][e] * (float)yv[p][e];
    }
  }
  const float rs = 1.f / sqrtf(wave_sum(ss) / (float)group + eps);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = (lane + 64 * p) * V;
    if (i < group) {
      const vec wv = *reinterpret_cast<const vec*>(w + i);
      vec o;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float zz = (float)zv[p][e], gate = 1.f / (1.f + __expf(-zz));
        o[e] = (T)((float)yv[p][e] * rs * (float)wv[e] * (sig ? gate : zz * gate));
      }
      *reinterpret_cast<vec*>(out + row * out_stride + g0 + i) = o;
    }
  }
}

// Any tap count 1 <= K <= 32, and an output that is the input (each thread reads a row before it writes
// it): one thread per channel walks its sequence.  KK > 0: that many taps, known at compile time, so that the window and
// the taps stay in registers (bf16; sums in the order of ssm_conv1d_kernel).  In place, runtime loops -> KK = 4:
// 4000 rows of 8192 channels in 3 sequences 827 -> 451 us, one of 500 rows of 4352 218 -> 101, 64 decode rows 11 either way.
template <typename T, int KK = 0>
__global__ __launch_bounds__(256) void ssm_conv1d_any_kernel(const T* __restrict__ x, int64_t x_stride,
                                                             const T* __restrict__ w, const T* __restrict__ bias,
                                                             T* __restrict__ out, int64_t out_stride,
                                                             T* __restrict__ state, const int* __restrict__ cu,
                                                             const int* __restrict__ slot, const int* __restrict__ reset,
                                                             int C, int taps) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (c >= C) return;
  const int r0 = cu[s], r1 = cu[s + 1];
  if (r1 <= r0) return;
  const int K = KK > 0 ? KK : taps;
  T* st = state + ((int64_t)slot[s] * C + c) * (K - 1);
  float win[KK > 0 ? KK : 31], wt[KK > 0 ? KK : 32];
  const bool fresh = reset[s] != 0;
  for (int j = 0; j < K - 1; ++j) win[j] = fresh ? 0.f : (float)st[j];
  for (int j = 0; j < K; ++j) wt[j] = (float)w[(int64_t)c * K + j];
  const float b = bias != nullptr ? (float)bias[c] : 0.f;
  for (int r = r0; r < r1; ++r) {
    const float v = (float)x[(int64_t)r * x_stride + c];
    float acc = b + wt[K - 1] * v;
    for (int j = 0; j < K - 1; ++j) acc += wt[j] * win[j];
    for (int j = 0; j + 1 < K - 1; ++j) win[j] = win[j + 1];
    if (K > 1) win[K - 2] = v;
    out[(int64_t)r * out_stride + c] = (T)(KK > 0 ? silu_f(acc) : acc / (1.f + expf(-acc)));
  }
  for (int j = 0; j < K - 1; ++j) st[j] = (T)win[j];
}

// Any head shape (P x N) and unaligned operand views: the fallback of ssm_scan_kernel, which needs
// 256 % P == 0, N / (256 / P) in {8, 16, 32, 64} and 16-byte aligned B / C rows.  One workgroup
// per (head, sequence); the head's fp32 state lives in LDS ([P][N + 1], or stays in global memory
// when it does not fit) for the whole sequence; per row: every thread updates its share of the
// P x N entries, then thread p reduces row p against C.  Two barriers per row.
template <typename T>
__global__ __launch_bounds__(256) void ssm_scan_any_kernel(
    const T* __restrict__ x, int64_t x_stride, const T* __restrict__ dt, int64_t dt_stride,
    const T* __restrict__ B, const T* __restrict__ Cm, int64_t bc_stride, const float* __restrict__ A,
    const float* __restrict__ D, const float* __restrict__ dt_bias, float dt_min, float* __restrict__ state,
    T* __restrict__ y, int64_t y_stride, const int* __restrict__ cu, const int* __restrict__ slot,
    const int* __restrict__ reset, int H, int P, int N, int G, int use_lds) {
  extern __shared__ float sm[];
  const int h = blockIdx.x, s = blockIdx.y;
  const int r0 = cu[s], r1 = cu[s + 1];
  if (r1 <= r0) return;
  const int g = h / (H / G);
  float* gst = state + ((int64_t)slot[s] * H + h) * P * N;
  float* st = use_lds ? sm : gst;
  const int ld = use_lds ? N + 1 : N;
  const int PN = P * N;
  const bool fresh = reset[s] != 0;
  if (use_lds || fresh)
    for (int e = threadIdx.x; e < PN; e += 256) st[(e / N) * ld + e % N] = fresh ? 0.f : gst[e];
  __syncthreads();
  const float a = A[h], d = D[h], db = dt_bias[h];
  for (int r = r0; r < r1; ++r) {
    const float dtr = (float)dt[(int64_t)r * dt_stride + h] + db;
    const float dtv = fmaxf(dtr > 20.f ? dtr : log1pf(expf(dtr)), dt_min);
    const float dA = expf(dtv * a);
    const T* xr = x + (int64_t)r * x_stride + h * P;
    const T* br = B + (int64_t)r * bc_stride + (int64_t)g * N;
    const T* cr = Cm + (int64_t)r * bc_stride + (int64_t)g * N;
    for (int e = threadIdx.x; e < PN; e += 256) {
      const int p = e / N, n = e - p * N;
      st[p * ld + n] = st[p * ld + n] * dA + dtv * (float)xr[p] * (float)br[n];
    }
    __syncthreads();
    for (int p = threadIdx.x; p < P; p += 256) {
      float acc = 0.f;
      for (int n = 0; n < N; ++n) acc += (float)cr[n] * st[p * ld + n];
      y[(int64_t)r * y_stride + h * P + p] = (T)(acc + d * (float)xr[p]);
    }
    __syncthreads();
  }
  if (use_lds)
    for (int e = threadIdx.x; e < PN; e += 256) gst[e] = st[(e / N) * ld + e % N];
}

}  // namespace

OME_API int ome_ssm_conv1d(const void* x, int64_t x_stride, const void* w, const void* bias, void* out,
                           int64_t out_stride, void* state, const int* cu, const int* slot, const int* reset, int S,
                           int T, int C, int K, int f32, hipStream_t stream) {
  if (S <= 0 || C <= 0) return 0;
  dim3 grid((C + 255) / 256, S);
  if (f32) {   // fp32 models: inputs, taps, outputs and the tail state are float
    if (K < 1 || K > 32) return -2;
    ssm_conv1d_any_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, x_stride, (const float*)w,
                                                           (const float*)bias, (float*)out, out_stride,
                                                           (float*)state, cu, slot, reset, C, K);
    OME_CHECK_LAUNCH();
    return 0;
  }
  // 16-byte pieces where every row and the taps allow them, single channels otherwise; an output that
  // overlaps the input (or lies between its rows), and more than 6 taps: the kernel that walks each sequence in order
  const bf16 *xb = (const bf16*)x, *ob = (const bf16*)out;
  const bool apart = T > 0 && (xb + (int64_t)(T - 1) * x_stride + C <= ob || ob + (int64_t)(T - 1) * out_stride + C <= xb);
  const bool vec8 = C % 8 == 0 && x_stride % 8 == 0 && out_stride % 8 == 0 &&
                    (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)out | (uintptr_t)state) & 15) == 0;
  const int lanes = vec8 ? C / 8 : C;
  const int by_seq = T <= S;
  const dim3 tiles(((by_seq ? 0 : T / CT) + S + 3) / 4, (lanes + 63) / 64);
#define CONV_CASE(KK)                                                                                                  \
  case KK:                                                                                                              \
    if (!apart || tiles.y > 65535)                                                                                      \
      ssm_conv1d_any_kernel<bf16, KK><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)w, (const bf16*)bias, \
                                                                (bf16*)out, out_stride, (bf16*)state, cu, slot, reset, C, K); \
    else if (vec8)                                                                                                      \
      ssm_conv1d_kernel<KK, 8><<<tiles, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)w, (const bf16*)bias,  \
                                                          (bf16*)out, out_stride, (bf16*)state, cu, slot, reset, S, C, by_seq); \
    else                                                                                                                \
      ssm_conv1d_kernel<KK, 1><<<tiles, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)w, (const bf16*)bias,  \
                                                          (bf16*)out, out_stride, (bf16*)state, cu, slot, reset, S, C, by_seq); \
    break;
  switch (K) {
    CONV_CASE(2)
    CONV_CASE(3)
    CONV_CASE(4)
    CONV_CASE(5)
    CONV_CASE(6)
    default:
      if (K < 1 || K > 32) return -2;
      ssm_conv1d_any_kernel<bf16><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)w, (const bf16*)bias,
                                                      (bf16*)out, out_stride, (bf16*)state, cu, slot, reset, C, K);
      break;
  }
#undef CONV_CASE
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_dyn_conv1d(const void* x, int64_t x_stride, const void* kern, int64_t k_stride, int cpk, void* out,
                           int64_t out_stride, void* state, const int* cu, const int* slot, const int* reset, int S,
                           int C, int K, hipStream_t stream) {
  if (S <= 0 || C <= 0) return 0;
  if (cpk <= 0 || C % cpk) return -3;
  dim3 grid((C + 255) / 256, S);
#define DCONV_CASE(KK)                                                                                         \
  case KK:                                                                                                      \
    dyn_conv1d_kernel<KK><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)kern, k_stride, cpk, \
                                                    (bf16*)out, out_stride, (bf16*)state, cu, slot, reset, C);   \
    break;
  switch (K) {
    DCONV_CASE(2)
    DCONV_CASE(3)
    DCONV_CASE(4)
    DCONV_CASE(5)
    DCONV_CASE(6)
    default:
      return -2;
  }
#undef DCONV_CASE
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_ssm_scan(const void* x, int64_t x_stride, const void* dt, int64_t dt_stride, const void* B,
                         const void* Cm, int64_t bc_stride, const float* A, const float* D, const float* dt_bias,
                         float dt_min, float* state, void* y, int64_t y_stride, const int* cu, const int* slot,
                         const int* reset, int S, int H, int P, int N, int G, int f32, hipStream_t stream) {
  if (S <= 0) return 0;
  if (P <= 0 || N <= 0 || G <= 0 || H % G != 0) return -2;
  {
    // the register-resident kernel needs its tiling (256 % P, 8 | N / (256 / P) <= 64) and B / C
    // rows it can read as 16-byte vectors; every other shape or view takes the generic kernel
    const int tp = 256 % P == 0 ? 256 / P : 0;
    const int np = tp > 0 && N % tp == 0 ? N / tp : 0;
    const bool fast = (np == 8 || np == 16 || np == 32 || np == 64) && bc_stride % 8 == 0 && N % 8 == 0 &&
                      ((uintptr_t)B % 16 == 0) && ((uintptr_t)Cm % 16 == 0) && ((uintptr_t)state % 16 == 0);
    if (!fast || f32) {
      const size_t need = (size_t)P * (N + 1) * sizeof(float);
      const int use_lds = need <= 64 * 1024;
      if (f32)
        ssm_scan_any_kernel<float><<<dim3(H, S), 256, use_lds ? need : 0, stream>>>(
            (const float*)x, x_stride, (const float*)dt, dt_stride, (const float*)B, (const float*)Cm, bc_stride, A,
            D, dt_bias, dt_min, state, (float*)y, y_stride, cu, slot, reset, H, P, N, G, use_lds);
      else
        ssm_scan_any_kernel<bf16><<<dim3(H, S), 256, use_lds ? need : 0, stream>>>(
            (const bf16*)x, x_stride, (const bf16*)dt, dt_stride, (const bf16*)B, (const bf16*)Cm, bc_stride, A, D,
            dt_bias, dt_min, state, (bf16*)y, y_stride, cu, slot, reset, H, P, N, G, use_lds);
      OME_CHECK_LAUNCH();
      return 0;
    }
  }
  // rows per workgroup: the whole head (PB = P).  Splitting a head's rows over more workgroups
  // (PB = P/4, 8 states per lane) measured SLOWER for 2 x 512-row prefill on gfx950 (812 vs 550 us,
  // scripts/ssm_scan_bench.py): the row loop is latency-bound per step, not occupancy-bound.
  const char* pbe = getenv("OME_SSM_PB");
  const int PB = pbe != nullptr && atoi(pbe) > 0 && P % atoi(pbe) == 0 ? atoi(pbe) : P;
  const int tpp = 256 / PB;
  if (N % tpp != 0) return -2;
  const int npt = N / tpp;
  dim3 grid(H * (P / PB), S);
#define SCAN_CASE(NN)                                                                                          \
  case NN:                                                                                                      \
    if (nt)                                                                                                     \
      ssm_scan_kernel<NN, true><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)dt, dt_stride,  \
                                                          (const bf16*)B, (const bf16*)Cm, bc_stride, A, D,      \
                                                          dt_bias, dt_min, state, (bf16*)y, y_stride, cu, slot,  \
                                                          reset, H, P, N, G, PB);                                \
    else                                                                                                        \
      ssm_scan_kernel<NN, false><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)dt, dt_stride, \
                                                           (const bf16*)B, (const bf16*)Cm, bc_stride, A, D,     \
                                                           dt_bias, dt_min, state, (bf16*)y, y_stride, cu, slot, \
                                                           reset, H, P, N, G, PB);                               \
    break;
  const char* nte = getenv("OME_SSM_NT");  // state I/O: 1 = non-temporal, 0 = plain (default)
  const bool nt = nte != nullptr && atoi(nte) != 0;
  switch (npt) {
    SCAN_CASE(8)
    SCAN_CASE(16)
    SCAN_CASE(32)
    SCAN_CASE(64)
    default:
      return -3;
  }
#undef SCAN_CASE
  OME_CHECK_LAUNCH();
  return 0;
}

OME_API int ome_gated_rmsnorm(const void* y, int64_t y_stride, const void* z, int64_t z_stride, const void* w,
                              void* out, int64_t out_stride, int rows, int I, int group, float eps,
                              int norm_first, int f32, hipStream_t stream) {
  // norm_first | 2: no intermediate rounding | 4: sigmoid gate (with 1 and 2)
  if (rows <= 0) return 0;
  if (group <= 0 || I % group != 0 || ((norm_first & 4) && (norm_first & 3) != 3)) return -2;
  const int64_t groups = (int64_t)rows * (I / group);
  if (!f32 && y_stride % 8 == 0 && z_stride % 8 == 0 && out_stride % 8 == 0 && groups <= (int64_t)4 * 0x7fffffff &&
      (((uintptr_t)y | (uintptr_t)z | (uintptr_t)w | (uintptr_t)out) & 15) == 0) {
#define GATED_VEC(L, N)                                                                                              \
  case 8 * (L) * (N):                                                                                                 \
    gated_rmsnorm_vec_kernel<L, N><<<(unsigned)((groups + 256 / (L) - 1) / (256 / (L))), 256, 0, stream>>>(           \
        (const bf16*)y, y_stride, (const bf16*)z, z_stride, (const bf16*)w, (bf16*)out, out_stride, groups, I / group, \
        eps, norm_first);                                                                                             \
    OME_CHECK_LAUNCH();                                                                                               \
    return 0;
    switch (group) {
      GATED_VEC(8, 1)
      GATED_VEC(16, 1)
      GATED_VEC(32, 1)
      GATED_VEC(64, 1)
      GATED_VEC(64, 2)
      GATED_VEC(64, 4)
    }
#undef GATED_VEC
  }
  if ((norm_first & 3) == 3 && group <= 512 && group % 2 == 0) {
    const int esz = f32 ? 4 : 2;
    auto al = [&](const void* p, int64_t stride) { return (((uintptr_t)p | (uintptr_t)(stride * esz)) & (2 * esz - 1)) == 0; };
    if (al(y, y_stride) && al(z, z_stride) && al(w, 0) && al(out, out_stride)) {
      const int per_row = I / group, sig = (norm_first & 4) != 0;
      const int64_t n = (int64_t)rows * per_row;
      if (n > (int64_t)4 * 0x7fffffff) return -3;
      const int nblk = (int)((n + 3) / 4);
      if (f32)
        gated_rmsnorm_wave_kernel<float, 2><<<nblk, 256, 0, stream>>>((const float*)y, y_stride, (const float*)z, z_stride,
                                                                      (const float*)w, (float*)out, out_stride, n, per_row,
                                                                      group, eps, sig);
      else
        gated_rmsnorm_wave_kernel<bf16, 2><<<nblk, 256, 0, stream>>>((const bf16*)y, y_stride, (const bf16*)z, z_stride,
                                                                     (const bf16*)w, (bf16*)out, out_stride, n, per_row, group,
                                                                     eps, sig);
      OME_CHECK_LAUNCH();
      return 0;
    }
  }
  dim3 grid(I / group, rows);
  if (f32)
    gated_rmsnorm_kernel<float><<<grid, 256, 0, stream>>>((const float*)y, y_stride, (const float*)z, z_stride,
                                                          (const float*)w, (float*)out, out_stride, group, eps,
                                                          norm_first);
  else
    gated_rmsnorm_kernel<bf16><<<grid, 256, 0, stream>>>((const bf16*)y, y_stride, (const bf16*)z, z_stride,
                                                         (const bf16*)w, (bf16*)out, out_stride, group, eps,
                                                         norm_first);
  OME_CHECK_LAUNCH();
  return 0;
}

// ------------------------------------------------------------------------------------------
// Residual causal convolution: out[r, c] = x[r, c] + sum_j w[c, j] * x[r - K + 1 + j, c]; x is an
// fp32 stream (TX = float) or a row already rounded to the taps' type (TX = T); sums are fp32
// (tap K-1 on the current row, zeros before a sequence's start, no bias, no activation), over a
// varlen batch; the last K-1 INPUT rows of every sequence live in `state` [slots, C, K-1] (fp32)
// between steps.  Not recurrent, so time is parallel: grid (channel blocks, sequences, row tiles of
// CM_TILE); a thread owns one channel of one tile and slides a register window over its rows.  Only
// a sequence's first tile touches the state: it reads the old tail before its rows and writes the
// new one (from the chunk's last rows, or from the old tail shifted when the chunk is shorter than
// K-1), so no other tile races with it.  Needs K - 1 <= CM_TILE.
// ------------------------------------------------------------------------------------------
namespace {
constexpr int CM_TILE = 64;

template <typename T, typename TX>
__global__ __launch_bounds__(256) void conv_mix_kernel(const TX* __restrict__ x, int64_t x_stride,
                                                       const T* __restrict__ w, T* __restrict__ out,
                                                       int64_t out_stride, float* __restrict__ state,
                                                       const int* __restrict__ cu, const int* __restrict__ slot,
                                                       const int* __restrict__ reset, int C, int K) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int s = blockIdx.y;
  const int r0 = cu[s], r1 = cu[s + 1];
  const int a = r0 + blockIdx.z * CM_TILE;
  if (c >= C || a >= r1) return;
  const int e = min(a + CM_TILE, r1);
  float win[31], wt[32];
  for (int j = 0; j < K; ++j) wt[j] = (float)w[(int64_t)c * K + j];
  if (blockIdx.z == 0) {
    float* st = state + ((int64_t)slot[s] * C + c) * (K - 1);
    const bool fresh = reset[s] != 0;
    for (int j = 0; j < K - 1; ++j) win[j] = fresh ? 0.f : st[j];
    const int L = r1 - r0;
    for (int j = 0; j < K - 1; ++j) {   // input index L - (K-1) + j of the chunk; negative = old tail
      const int i = L - (K - 1) + j;
      st[j] = i >= 0 ? (float)x[(int64_t)(r0 + i) * x_stride + c] : win[K - 1 + i];
    }
  } else {
    for (int j = 0; j < K - 1; ++j) win[j] = (float)x[(int64_t)(a - (K - 1) + j) * x_stride + c];
  }
  for (int r = a; r < e; ++r) {
    const float v = (float)x[(int64_t)r * x_stride + c];
    float acc = v + wt[K - 1] * v;
    for (int j = 0; j < K - 1; ++j) acc += wt[j] * win[j];
    for (int j = 0; j + 1 < K - 1; ++j) win[j] = win[j + 1];
    if (K > 1) win[K - 2] = v;
    out[(int64_t)r * out_stride + c] = (T)acc;
  }
}
}  // namespace

OME_API int ome_conv_mix(const void* x, int64_t x_stride, const void* w, void* out, int64_t out_stride, float* state,
                         const int* cu, const int* slot, const int* reset, int S, int T, int C, int K, int f32,
                         int x_f32, hipStream_t stream) {
  if (S <= 0 || C <= 0 || T <= 0) return 0;
  if (K < 1 || K > 32) return -2;
  const int tiles = (T + CM_TILE - 1) / CM_TILE;
  if (tiles > 65535 || S > 65535) return -3;
  dim3 grid((C + 255) / 256, S, tiles);
  if (f32)
    conv_mix_kernel<float, float><<<grid, 256, 0, stream>>>((const float*)x, x_stride, (const float*)w, (float*)out,
                                                            out_stride, state, cu, slot, reset, C, K);
  else if (x_f32)
    conv_mix_kernel<bf16, float><<<grid, 256, 0, stream>>>((const float*)x, x_stride, (const bf16*)w, (bf16*)out,
                                                           out_stride, state, cu, slot, reset, C, K);
  else
    conv_mix_kernel<bf16, bf16><<<grid, 256, 0, stream>>>((const bf16*)x, x_stride, (const bf16*)w, (bf16*)out,
                                                          out_stride, state, cu, slot, reset, C, K);
  OME_CHECK_LAUNCH();
  return 0;
}
