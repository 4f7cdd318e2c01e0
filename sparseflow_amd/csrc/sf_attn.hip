// Fused spike-driven self-attention core (no softmax):
//   y[tb, m, h, :] = scale * sum_d q[tb, m, h, d] * KV[tb, h, d, :],
//   KV[tb, h, d, e] = sum_j k[tb, j, h, d] * v[tb, j, h, e]
// which equals (q @ k^T * scale) @ v of the reference's attention stages
// (Kernels/attention.py:27-121 over Kernels/bmm.py) without the seq x seq
// score matrix: per (frame, head) the kernel reads q, k and v once and
// writes y once.
//
// Both products run on the matrix cores in f32 (32x32x2, for D = 16
// 16x16x4: full f32 products and sums, for spikes and any other values),
// straight from global memory: a K step of the first product is one row of
// k and of v per half wavefront (two 128-byte runs per load at D = 32), and
// KV, as the first product leaves it in the accumulators (lane = column e,
// register = row d), is the second product's B operand as it stands, with
// q's four-element pieces as the A operand.  q, k and v are not staged in LDS,
// and the loads of the next K steps and of the next rows of q are in flight
// during the MFMAs.  With enough items a wavefront takes one and waits for no
// other; with few, four wavefronts share an item's rows and add their partial
// sums of KV through LDS, behind the one barrier.  q elements below the
// activity cutoff count as zero (the reference's prescan test on the left
// operand).  Sums run in an order fixed by the shape: deterministic.
//
// Bound by HBM (q, k, v in, y out).  At 256 frames x 12 heads x 196 tokens x
// 32 (308 MB), inputs new at every call: 64 us = 4.8 TB/s, the card's copy rate
// (the same inputs again, partly in the last-level cache: 52-57 us); the form
// before it, which staged k and v in LDS as f32 and formed KV and the rows on
// the VALU, took 127 us.
//
// An item whose KV is not finite everywhere takes its q rows' active elements
// one by one instead: there an inactive one must not meet a KV row (0 * inf
// would be NaN).
//
// Layout: element (tb, m, h, d) at tb*s_tb + m*s_m + h*s_h + d for q, k, v
// (one set of strides) and for y (its own), so both token-major
// [TB, S, H, D] (the projections' output) and head-major [TB, H, S, D]
// tensors are read in place.
#include "sf_tile.h"

namespace sf {

namespace {

constexpr int kAttnWaves = 4;  // wavefronts per workgroup
constexpr int kAttnItemsPerCu = 8;  // items per CU from which a wavefront takes a whole item

template <int MT> struct AttnAcc;
template <> struct AttnAcc<32> { typedef float type __attribute__((ext_vector_type(16))); };
template <> struct AttnAcc<16> { typedef float type __attribute__((ext_vector_type(4))); };

template <int MT>
__device__ __forceinline__ typename AttnAcc<MT>::type attn_mfma(float a, float b, typename AttnAcc<MT>::type c) {
  if constexpr (MT == 32) return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four consecutive elements (one load when VEC: p is then aligned to 4
// elements).
template <typename T, bool VEC>
__device__ __forceinline__ void attn_load4(const T* __restrict__ p, float (&v)[4]) {
  if constexpr (VEC) {
    struct alignas(4 * sizeof(T)) Q4 { T e[4]; };
    const Q4 q = *reinterpret_cast<const Q4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = to_f32<T>(q.e[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = to_f32<T>(p[i]);
  }
}

// W wavefronts share an item's K rows and q rows (1: a wavefront per item).
template <typename T, typename TOut, int D, int W, bool VEC>
__global__ __launch_bounds__(64 * kAttnWaves) void k_spike_attn(AttnArgs a) {
  constexpr int MT = D == 16 ? 16 : 32;  // MFMA tile edge
  constexpr int NB = D / MT;             // tiles along D
  constexpr int KS = 64 / MT;            // rows of k, v per K step
  constexpr int NR = MT * MT / 64;       // accumulator registers per tile
  constexpr int NG = NR / 4;             // four-element pieces of q per tile row and lane
  constexpr int U = NB == 2 ? 4 : 8;     // K steps per batch of loads
  typedef typename AttnAcc<MT>::type Acc;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane % MT, kk = lane / MT;
  const int S = a.s;
  const int64_t items = a.tb * (int64_t)a.h;
  const int64_t item = a.item0 + (W == 1 ? (int64_t)blockIdx.x * kAttnWaves + wave : (int64_t)blockIdx.x);
  const int part = W == 1 ? 0 : wave;
  if (item >= items) return;  // W == 1 only: a whole wavefront, and no barrier follows there
  const int64_t tbi = item / a.h;
  const int hh = (int)(item - tbi * a.h);
  const int64_t base = tbi * a.s_tb + hh * a.s_h;
  const int64_t ybase = tbi * a.y_tb + hh * a.y_h;
  const T* __restrict__ Q = static_cast<const T*>(a.q) + base;
  const T* __restrict__ K = static_cast<const T*>(a.k) + base;
  const T* __restrict__ V = static_cast<const T*>(a.v) + base;
  TOut* __restrict__ Y = static_cast<TOut*>(a.y) + ybase;

  // ---- KV = k^T v ----
  Acc kv[NB][NB];
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int eb = 0; eb < NB; ++eb)
#pragma unroll
      for (int i = 0; i < NR; ++i) kv[db][eb][i] = 0.f;
  constexpr int RB = U * KS;  // rows per batch
  const int batches = (S + RB - 1) / RB;
  T kr[U][NB], vr[U][NB];
  auto fetch = [&](int b) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // Rows past the end read the last one; they are zeroed below.
      const int64_t off = (int64_t)min(b * RB + u * KS + kk, S - 1) * a.s_m + n;
#pragma unroll
      for (int db = 0; db < NB; ++db) {
        kr[u][db] = K[off + db * MT];
        vr[u][db] = V[off + db * MT];
      }
    }
  };
  if (part < batches) fetch(part);
  for (int b = part; b < batches; b += W) {
    float kf[U][NB], vf[U][NB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = b * RB + u * KS + kk < S;
#pragma unroll
      for (int db = 0; db < NB; ++db) {
        kf[u][db] = in ? to_f32<T>(kr[u][db]) : 0.f;
        vf[u][db] = in ? to_f32<T>(vr[u][db]) : 0.f;
      }
    }
    if (b + W < batches) fetch(b + W);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int eb = 0; eb < NB; ++eb) kv[db][eb] = attn_mfma<MT>(kf[u][db], vf[u][eb], kv[db][eb]);
  }
  if constexpr (W > 1) {
    // The wavefronts' partial sums, added in their order by every one.
    __shared__ float s_part[W][NB * NB * NR][64];
#pragma unroll
    for (int t = 0; t < NB * NB; ++t)
#pragma unroll
      for (int i = 0; i < NR; ++i) s_part[part][t * NR + i][lane] = kv[t / NB][t % NB][i];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NB * NB; ++t)
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        float s = s_part[0][t * NR + i][lane];
#pragma unroll
        for (int w = 1; w < W; ++w) s += s_part[w][t * NR + i][lane];
        kv[t / NB][t % NB][i] = s;
      }
  }
  // Lane (n, kk) holds KV[d][e], e = eb * MT + n, in kv[d / MT][eb][r] for
  // the d whose place in its tile is 8 (r / 4) + 4 kk + r % 4 (MT = 32) or
  // 4 kk + r (MT = 16).
  bool bad = false;
#pragma unroll
  for (int t = 0; t < NB * NB; ++t)
#pragma unroll
    for (int i = 0; i < NR; ++i) bad |= !(fabsf(kv[t / NB][t % NB][i]) < __builtin_huge_valf());

  if (__ballot(bad) != 0ull) {
    // ---- rows of q by their active elements ----
    constexpr int R = 64 / D;
    const int r = lane / D, e = lane % D;
    for (int m0 = part * R; m0 < S; m0 += W * R) {
      const int m = m0 + r, mc = min(m, S - 1);
      float sum = 0.f;
      int e_t = e;  // opaque, so that KV's D rows are not exchanged ahead of the loop into D registers
      asm volatile("" : "+v"(e_t));
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int dd = d % MT;
        const int reg = MT == 32 ? 4 * (dd / 8) + dd % 4 : dd % 4;
        const int src = (MT == 32 ? (dd / 4) % 2 : dd / 4) * MT + e_t % MT;
        float w = __shfl(kv[d / MT][0][reg], src, 64);
        if constexpr (NB == 2) {
          const float w1 = __shfl(kv[d / MT][1][reg], src, 64);
          w = e_t >= MT ? w1 : w;
        }
        const float qd = to_f32<T>(Q[(int64_t)mc * a.s_m + d]);
        if (fabsf(qd) >= a.cutoff) sum = fmaf(qd, w, sum);
      }
      if (m < S) Y[(int64_t)m * a.y_m + e] = from_f32<TOut>(sum * a.scale);
    }
    return;
  }

  // ---- y = q KV: MT rows of q per tile ----
  const int tiles = (S + MT - 1) / MT;
  float qn[NB][NG][4];
  auto fetch_q = [&](int t) {
    const T* __restrict__ row = Q + (int64_t)min(t * MT + n, S - 1) * a.s_m + 4 * kk;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int g = 0; g < NG; ++g) attn_load4<T, VEC>(row + db * MT + 8 * g, qn[db][g]);
  };
  if (part < tiles) fetch_q(part);
  for (int t = part; t < tiles; t += W) {
    float qc[NB][NG][4];
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float q = qn[db][g][i];
          qc[db][g][i] = fabsf(q) >= a.cutoff ? q : 0.f;
        }
    if (t + W < tiles) fetch_q(t + W);
#pragma unroll
    for (int eb = 0; eb < NB; ++eb) {
      Acc y;
#pragma unroll
      for (int i = 0; i < NR; ++i) y[i] = 0.f;
#pragma unroll
      for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i) y = attn_mfma<MT>(qc[db][g][i], kv[db][eb][4 * g + i], y);
      // Register i: row 8 (i / 4) + 4 kk + i % 4 (MT = 32) or 4 kk + i of the
      // tile, column eb * MT + n.
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int m = t * MT + 8 * (i / 4) + 4 * kk + i % 4;
        if (m < S) Y[(int64_t)m * a.y_m + eb * MT + n] = from_f32<TOut>(y[i] * a.scale);
      }
    }
  }
}

template <typename T, typename TOut, int D, int W>
int launch_attn_w(AttnArgs a, hipStream_t stream) {
  // q's four-element loads: its base and row starts at multiples of them.
  const bool vec = ((reinterpret_cast<uintptr_t>(a.q) / sizeof(T)) | (uintptr_t)(a.s_tb | a.s_m | a.s_h)) % 4 == 0;
  // (A launch holds fewer than 2^32 threads.)
  constexpr int64_t kLaunchItems = (int64_t)1 << 24;
  const int64_t items = a.tb * (int64_t)a.h;
  for (a.item0 = 0; a.item0 < items; a.item0 += kLaunchItems) {
    const int64_t n = items - a.item0 < kLaunchItems ? items - a.item0 : kLaunchItems;
    const dim3 grid((unsigned)(W == 1 ? (n + kAttnWaves - 1) / kAttnWaves : n)), block(64 * kAttnWaves);
    if (vec) hipLaunchKernelGGL((k_spike_attn<T, TOut, D, W, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((k_spike_attn<T, TOut, D, W, false>), grid, block, 0, stream, a);
    const int rc = (int)hipGetLastError();
    if (rc != (int)hipSuccess) return rc;
  }
  return (int)hipSuccess;
}

template <typename T, typename TOut, int D>
int launch_attn_t(const AttnArgs& a, hipStream_t stream) {
  // A wavefront per item once there are enough items to fill the CUs with
  // them; a workgroup per item below (2 to 12 items a CU differ by under 5%, at
  // 12 in favour of the first, whose partial sums cost nothing, while a few
  // items on single wavefronts leave most of the GPU idle).
  return a.tb * (int64_t)a.h >= (int64_t)num_cus() * kAttnItemsPerCu ? launch_attn_w<T, TOut, D, 1>(a, stream)
                                                                     : launch_attn_w<T, TOut, D, kAttnWaves>(a, stream);
}

template <typename T, typename TOut>
int launch_attn_o(const AttnArgs& a, hipStream_t stream) {
  switch (a.d) {
    case 16: return launch_attn_t<T, TOut, 16>(a, stream);
    case 32: return launch_attn_t<T, TOut, 32>(a, stream);
    default: return launch_attn_t<T, TOut, 64>(a, stream);
  }
}

template <typename T>
int launch_attn_d(const AttnArgs& a, int out_dtype, hipStream_t stream) {
  if (out_dtype == SF_F32) return launch_attn_o<T, float>(a, stream);
  return launch_attn_o<T, T>(a, stream);
}

}  // namespace

// Head widths of the matrix cores' tiles.  The lengths are the declared range of
// the entry point; the kernel itself has no limit on them.
int attn_max_tokens(int d) { return d == 16 ? 1271 : d == 32 ? 623 : d == 64 ? 287 : 0; }

int launch_spike_attn(const AttnArgs& a, int in_dtype, int out_dtype, hipStream_t stream) {
  timing_begin(K_ATTN, stream);
  const int rc = in_dtype == SF_F16    ? launch_attn_d<__half>(a, out_dtype, stream)
                 : in_dtype == SF_BF16 ? launch_attn_d<__hip_bfloat16>(a, out_dtype, stream)
                                       : launch_attn_d<float>(a, out_dtype, stream);
  timing_end(K_ATTN, stream);
  return rc;
}

}  // namespace sf
