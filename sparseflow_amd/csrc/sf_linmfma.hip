// Sparse Linear on the matrix cores: y[m, c_out] = x[m, k] @ W^T + bias at
// transformer spike densities (p ~ 0.1), where every 32-wide slice of K is
// live in some row of a tile and a VALU walk over the spikes loses to MFMA.
//
// Exactness without fp32 MFMA: W is split on the host into bf16 hi + lo
// parts (W = hi + lo + O(2^-17 |W|)) and x in the kernel (x = xh + xl; xl is
// zero for spikes and small integers), and y = xh @ hi^T + xh @ lo^T +
// xl @ hi^T carries ~16 bits of both operands.  Elements with f16(|x|) <=
// f16(threshold) count as zero, as in the prescan.
//
// One workgroup (4 wavefronts, 2 x 2) computes a 128-row x 128-column tile;
// each wavefront 64 x 64 = 4 x 4 MFMA 16x16x32 bf16 tiles (64 f32
// accumulators per lane).  K is walked in 32-wide steps: the x tile (128 x
// 32, converted to bf16 in registers) and the W tiles (128 columns x 32 of
// the [c_out][kp] bf16 hi and lo rows, from L2) are staged in LDS,
// double-buffered with one barrier per step; the next step's loads are in
// flight during the current step's MFMAs.  The main walk computes xh @ hi^T
// + xh @ lo^T and notes whether any staged element of x has a non-zero xl;
// only a workgroup that saw one walks K a second time for xl @ hi^T (for
// spikes, the transformer case, the third product is never formed).  The
// MFMAs of a walk run unconditionally: a data-dependent branch around them
// makes the compiler copy the 64 accumulators between AGPRs and VGPRs every
// step, which costs more than the products it would skip (an all-zero 128 x
// 32 slice of x is vanishingly rare at these densities; the spike walk
// serves sparse inputs).
// Row blocks are the slow index of the grid and workgroups are placed
// XCD-locally, so the column blocks of one row block run together on one
// XCD and share its x tile through that XCD's L2.
//
// Replaces the reference's sparse_linear_grouped_kernel (Kernels/linear.py:
// 360-457: fp16 tl.dot over active groups, dense tiles when all groups are
// live) for such inputs.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "sf_tile.h"

namespace sf {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kLmRows = 128;        // rows per workgroup tile
constexpr int kLmCols = 128;        // output columns per workgroup tile
constexpr int kLmK = 32;            // K per step
constexpr int kLmLda = kLmK;        // LDS row: 32 bf16 = 64 B, four 16-byte pieces
// 16-byte piece p of tile row r sits at piece p ^ ((r >> 1) & 3) of its
// row.  Measured on gfx950 (rocprofv3 SQ_LDS_BANK_CONFLICT over the
// kernel's ds_read_b128 fragment reads and ds_write_b128 staging writes):
// with 64-byte rows this swizzle is conflict-free for both, while the
// swizzle by (r >> 2) & 3 -- which also covers every bank once per 16 lanes
// -- costs a third more LDS cycles on the reads and doubles the writes.
__device__ __forceinline__ int lm_piece(int r, int p) { return p ^ ((r >> 1) & 3); }
constexpr int kLmMaxK = 8192;

__device__ __forceinline__ uint16_t bf16_bits(float f) {
  const __hip_bfloat16 h = __float2bfloat16(f);  // round to nearest even
  uint16_t u;
  __builtin_memcpy(&u, &h, 2);
  return u;
}

__device__ __forceinline__ float bf16_value(uint16_t u) {
  return __uint_as_float((uint32_t)u << 16);
}

// 16 consecutive elements of row `row` from column kk0, without branches
// and without touching the loaded values: out-of-range rows and columns
// load a valid element, and the count of valid elements (0..16) is returned
// for the staging to zero the rest -- any use of the values here would make
// the compiler wait for the loads before the MFMAs they are meant to
// overlap.  VEC: f32 input, k % 16 == 0 and x 16-byte aligned, so a
// 16-element run is entirely inside or entirely past the row.
template <typename TIn, bool VEC>
__device__ __forceinline__ int lm_load_x(const TIn* __restrict__ x, int64_t m, int k, int row, int kk0,
                                         float (&v)[16]) {
  const bool row_ok = row < m;
  const int64_t rr = row_ok ? row : 0;
  const int valid = row_ok ? min(max(k - kk0, 0), 16) : 0;
  if constexpr (VEC) {
    const float4* p = reinterpret_cast<const float4*>(x + rr * k + (valid > 0 ? kk0 : 0));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 t = p[q];
      v[4 * q] = t.x;
      v[4 * q + 1] = t.y;
      v[4 * q + 2] = t.z;
      v[4 * q + 3] = t.w;
    }
  } else {
    // Raw 16-bit or 32-bit elements; converted in the staging.
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const TIn t = x[rr * k + (j < valid ? kk0 + j : 0)];
      if constexpr (sizeof(TIn) == 4) {
        v[j] = t;
      } else {
        uint16_t u;
        __builtin_memcpy(&u, &t, 2);
        v[j] = __uint_as_float((uint32_t)u);  // bit pattern carried in a float register
      }
    }
  }
  return valid;
}

template <typename TIn, bool VEC>
__device__ __forceinline__ float lm_value(float raw) {
  if constexpr (VEC || sizeof(TIn) == 4) {
    return raw;
  } else {
    const uint16_t u = (uint16_t)__float_as_uint(raw);
    TIn t;
    __builtin_memcpy(&t, &u, 2);
    return to_f32<TIn>(t);
  }
}

// Stores a wavefront's 64 x 64 accumulator tile (acc[rt][ct] element i of
// lane l: row 16 rt + 4 (l >> 4) + i, column 16 ct + (l & 15)) plus the bias
// as rows of 16-byte pieces: each 16-row slice goes through the wavefront's
// own LDS region (16 rows of 68 floats: conflict-free both ways) and is read
// back as four consecutive columns per lane, so that one store instruction
// writes four 256-byte row runs (4-byte stores scattered over the rows
// wrote y at ~1.4 TB/s).  r_0, c_0: the tile's first row and column in y.
template <typename TOut>
__device__ __forceinline__ void lm_store_tile(const f32x4 (&acc)[4][4], float* __restrict__ stile,
                                              const float* __restrict__ bias, TOut* __restrict__ Y, int64_t m,
                                              int c_out, int64_t r_0, int c_0, int lane) {
  constexpr int kS = 68;  // floats per staged row
  const int g = lane >> 4, li = lane & 15;
  float bv[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const int col = c_0 + 16 * ct + li;
    bv[ct] = bias != nullptr && col < c_out ? bias[col] : 0.f;
  }
  const int rq = lane >> 4, cq = 4 * (lane & 15);  // read-back: rows rq + 4 j, columns cq .. cq + 3
  const int col = c_0 + cq;
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) stile[(4 * g + i) * kS + 16 * ct + li] = acc[rt][ct][i] + bv[ct];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's writes are done before its reads
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t row = r_0 + 16 * rt + rq + 4 * j;
      const float4 v = *reinterpret_cast<const float4*>(&stile[(rq + 4 * j) * kS + cq]);
      if (row < m && col < c_out) store4<TOut>(Y + row * c_out + col, v.x, v.y, v.z, v.w);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // its reads are done before the next slice's writes
  }
}

template <typename TIn, typename TOut, bool VEC>
__global__ __launch_bounds__(256) void k_linear_mfma(LinMfmaArgs a) {
  // Double-buffered LDS tiles (bf16 bit patterns): x [128 rows][32] (its hi
  // part in the main walk, its lo part in the second), W hi / lo [128
  // columns][32]; 48 KB, in one array (the output staging reuses it).
  __shared__ __align__(16) uint16_t s_tiles[3][2][kLmRows * kLmLda];
  auto& s_xh = s_tiles[0];
  auto& s_wh = s_tiles[1];
  auto& s_wl = s_tiles[2];
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const int ncb = (a.c_out + kLmCols - 1) / kLmCols;
  // The column blocks of a row block share its x tile through L2, which is
  // per XCD: placed XCD-locally, consecutive tiles run on one XCD.
  const int bid = xcd_range_block((int)blockIdx.x, (int)gridDim.x);
  const int64_t rb = bid / ncb;
  const int cb = (int)(bid - rb * ncb);
  const int64_t r0 = rb * kLmRows;
  const int c0 = cb * kLmCols;
  const int nsteps = a.kp / kLmK;
  const TIn* __restrict__ X = static_cast<const TIn*>(a.x);

  // Staging: thread t takes x row t / 2 and W column t / 2 of the tile, 16
  // k values at 16 * (t & 1).  Columns past c_out stage W row 0 (never stored).
  const int sr = tid >> 1, sh = tid & 1;
  const int wcol = c0 + sr < a.c_out ? c0 + sr : 0;
  const uint4* wh_src = reinterpret_cast<const uint4*>(a.wh + (int64_t)wcol * a.kp + 16 * sh);
  const uint4* wl_src = reinterpret_cast<const uint4*>(a.wl + (int64_t)wcol * a.kp + 16 * sh);
  float v[16];
  int v_valid = 0;
  uint4 wh0, wh1, wl0, wl1;
  // LO = false: the main walk (x hi, W hi and lo); LO = true: the second walk
  // (x lo, W hi).
  auto load_step = [&](int step, auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    const int kb = step * kLmK;  // 16-byte units: kb / 8
    wh0 = wh_src[kb / 8];
    wh1 = wh_src[kb / 8 + 1];
    if constexpr (!LO) {
      wl0 = wl_src[kb / 8];
      wl1 = wl_src[kb / 8 + 1];
    }
    v_valid = lm_load_x<TIn, VEC>(X, a.m, a.k, (int)(r0 + sr), kb + 16 * sh, v);  // r0 + sr < 2^30 + 128
  };
  bool inexact = false;  // some staged element of x has a non-zero lo part
  auto stage = [&](int buf, auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    uint32_t hx[8];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float t = lm_value<TIn, VEC>(v[j]);
      v[j] = (j < v_valid && fabsf(t) >= a.cutoff) ? t : 0.f;  // range, then the prescan's activity test
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint16_t h0 = bf16_bits(v[2 * j]), h1 = bf16_bits(v[2 * j + 1]);
      const float r0v = v[2 * j] - bf16_value(h0), r1v = v[2 * j + 1] - bf16_value(h1);
      if constexpr (LO) {
        hx[j] = (uint32_t)bf16_bits(r0v) | ((uint32_t)bf16_bits(r1v) << 16);
      } else {
        inexact |= (r0v != 0.f) | (r1v != 0.f);
        hx[j] = (uint32_t)h0 | ((uint32_t)h1 << 16);
      }
    }
    const int p0 = 8 * lm_piece(sr, 2 * sh), p1 = 8 * lm_piece(sr, 2 * sh + 1);  // bf16 offsets
    uint16_t* rx = &s_xh[buf][sr * kLmLda];
    uint16_t* rwh = &s_wh[buf][sr * kLmLda];
    *reinterpret_cast<uint4*>(rx + p0) = make_uint4(hx[0], hx[1], hx[2], hx[3]);
    *reinterpret_cast<uint4*>(rx + p1) = make_uint4(hx[4], hx[5], hx[6], hx[7]);
    *reinterpret_cast<uint4*>(rwh + p0) = wh0;
    *reinterpret_cast<uint4*>(rwh + p1) = wh1;
    if constexpr (!LO) {
      uint16_t* rwl = &s_wl[buf][sr * kLmLda];
      *reinterpret_cast<uint4*>(rwl + p0) = wl0;
      *reinterpret_cast<uint4*>(rwl + p1) = wl1;
    }
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int g = lane >> 4, li = lane & 15;
  // One walk over K: per step, x [128 x 32] times W^T [32 x 128] as the
  // products of the staged x tile with the staged W hi (and, in the main
  // walk, W lo) tiles.
  auto walk = [&](auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    load_step(0, lo_walk);
    stage(0, lo_walk);
    __syncthreads();
    for (int step = 0; step < nsteps; ++step) {
      const int buf = step & 1;
      // Next step's tiles are in flight during this step's MFMAs; the staging
      // after them is their first use.
      if (step + 1 < nsteps) load_step(step + 1, lo_walk);
      // Keep the scheduler from pulling the staging math (which waits for
      // those loads) above the MFMAs.
      __builtin_amdgcn_sched_barrier(0);
      {
        bf16x8 ax[4], bh[4], bl[4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          const int r = 64 * wc + 16 * ct + li;
          const int c = r * kLmLda + 8 * lm_piece(r, g);
          bh[ct] = *reinterpret_cast<const bf16x8*>(&s_wh[buf][c]);
          if constexpr (!LO) bl[ct] = *reinterpret_cast<const bf16x8*>(&s_wl[buf][c]);
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const int r = 64 * wr + 16 * rt + li;
          ax[rt] = *reinterpret_cast<const bf16x8*>(&s_xh[buf][r * kLmLda + 8 * lm_piece(r, g)]);
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int ct = 0; ct < 4; ++ct)
            acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[rt], bh[ct], acc[rt][ct], 0, 0, 0);
        if constexpr (!LO) {
#pragma unroll
          for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
              acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[rt], bl[ct], acc[rt][ct], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (step + 1 < nsteps) stage(buf ^ 1, lo_walk);
      __syncthreads();
    }
  };
  walk(std::false_type{});
  // Every staged element's lo part was zero in every thread: done (the
  // barrier's result is the same in every wavefront, so the branch is
  // uniform).
  if (__syncthreads_or(inexact ? 1 : 0)) walk(std::true_type{});

  // The last step's barrier: every wavefront is done with the tiles.
  float* stile = reinterpret_cast<float*>(&s_tiles[0][0][0]) + wave * (16 * 68);
  lm_store_tile<TOut>(acc, stile, a.bias, static_cast<TOut*>(a.y), a.m, a.c_out, r0 + 64 * wr, c0 + 64 * wc, lane);
}

// ---- the same product over the prescan's row bitmap --------------------
//
// For spike inputs the x tile is one bit per element: a lane's A fragment
// (8 consecutive k of one row) is one byte of that row's bitmap word, its
// bits turned into bf16 0 / 1 values on the VALU, so x costs 4 bytes per row
// per 32-wide K step instead of 128 (f32) and needs no staging.  A
// workgroup of 4 wavefronts computes one 256 x 128 tile, each wavefront
// 128 x 64 (8 x 4 MFMA tiles: a step's 8 W fragment reads serve 64
// products); per step the W tiles (bf16 hi and lo, 16 KB) and the rows'
// bitmap words (1 KB) go from global memory straight into a ring of three
// LDS buffers, requested two steps ahead and waited for by count.
// The barrier that ends a step waits for no load (in-kernel timestamps of a
// __syncthreads() version showed every step waiting for all of them), and
// 66.5 KB of LDS let two workgroups share a CU: their barriers are
// independent, so one's fragment reads and waits overlap the other's
// MFMAs, and a finished workgroup's stores drain while the next one on the
// CU starts (a persistent version with one 8-wavefront workgroup per CU
// stored every tile in lockstep on all CUs, ~6 us a round with the matrix
// cores idle).  Row blocks whose non-binary flag is set (a value other than 0 and
// 1 in some row) read their x tiles instead: A fragments from x split into
// bf16 hi + lo, three products per step (the exactness of the direct
// kernel).
// Barrier for LDS hand-offs: this wavefront's LDS accesses are complete
// before it, and the compiler moves no memory access across it.  Unlike
// __syncthreads() (whose release fence waits for every outstanding load,
// the direct LDS loads included) it leaves the loads of later steps in
// flight; their consumers wait for them by count.
__device__ __forceinline__ void ws_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr int kLbRows = 256;    // rows per workgroup tile
constexpr int kLbWaves = 4;
constexpr int kLbRT = 8;        // 16-row MFMA tiles per wavefront (128 rows)
constexpr int kLbBufs = 3;      // stage buffers (W tiles and words of one 32-wide K step)

// W tiles of step s (both parts) into LDS buffers (sh, sl) with direct
// loads: 1 KB blocks, wavefront w loading blocks 4 w .. 4 w + 3 (blocks 0..7
// the hi part, 8..15 the lo part); LDS position q of a part holds row q >> 2,
// stored piece q & 3, i.e. logical piece lm_piece(row, q & 3) (lm_piece is
// its own inverse).  Rows past c_out load row 0 (never stored).
__device__ __forceinline__ void lb_load_w(uint16_t* __restrict__ sh, uint16_t* __restrict__ sl,
                                          const uint16_t* __restrict__ wh, const uint16_t* __restrict__ wl, int kp,
                                          int c0, int c_out, int s, int wave, int lane) {
#pragma unroll
  for (int j = 0; j < 16 / kLbWaves; ++j) {
    const int u = (16 / kLbWaves) * wave + j;
    const int q = (u & 7) * 64 + lane;
    const int r = q >> 2;
    const int p = lm_piece(r, q & 3);
    const int col = c0 + r < c_out ? c0 + r : 0;
    const uint16_t* src = (u < 8 ? wh : wl) + (int64_t)col * kp + 32 * s + 8 * p;
    uint16_t* dst = (u < 8 ? sh : sl) + (u & 7) * 512;  // 1 KB = 512 bf16
    lds_dma16(src, dst);
  }
}
constexpr int kLbLoads = 16 / kLbWaves + 1;  // direct loads per wavefront and step (W blocks, words)

// Eight spikes (bits 0..7 of byte) as bf16 0 / 1 values, element i = bit i.
__device__ __forceinline__ bf16x8 spike_bf16x8(uint32_t byte) {
  uint32_t p[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    p[j] = (((byte >> (2 * j)) & 1u) * 0x3F80u) | (((byte >> (2 * j + 1)) & 1u) * 0x3F800000u);
  return __builtin_bit_cast(bf16x8, make_uint4(p[0], p[1], p[2], p[3]));
}

// A wavefront's (16 RT) x 64 tile as rows of 16-byte pieces (lm_store_tile's
// staging) through buffer stores: rows past m and columns past c_out fall
// outside the buffer range and are dropped.  The whole offset rides in the
// VGPR, soffset stays 0 (with an SGPR soffset the compiler adds no wait
// state between a 16-byte store and a VALU write of its data registers, and
// on gfx950 the last lanes of each 16-lane group then store the overwritten
// value).
template <int RT, typename TOut>
__device__ __forceinline__ void lb_store_tile(const f32x4 (&acc)[RT][4], float* __restrict__ stile,
                                              const float* __restrict__ bias, __amdgpu_buffer_rsrc_t ry, int64_t m,
                                              int c_out, int64_t r_0, int c_0, int lane) {
  constexpr int kS = 68;
  const int g = lane >> 4, li = lane & 15;
  float bv[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const int col = c_0 + 16 * ct + li;
    bv[ct] = bias != nullptr && col < c_out ? bias[col] : 0.f;
  }
  const int rq = lane >> 4, cq = 4 * (lane & 15);
  const int col = c_0 + cq;
  constexpr uint32_t B = (uint32_t)sizeof(TOut);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) stile[(4 * g + i) * kS + 16 * ct + li] = acc[rt][ct][i] + bv[ct];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t row = r_0 + 16 * rt + rq + 4 * j;
      const float4 v = *reinterpret_cast<const float4*>(&stile[(rq + 4 * j) * kS + cq]);
      int vo = (row < m && col < c_out) ? (int)((uint32_t)(row * c_out + col) * B) : 0x7fffffff;
      asm volatile("" : "+v"(vo));
      if constexpr (sizeof(TOut) == 4) {
        const sf_u32x4 q = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
        __builtin_amdgcn_raw_buffer_store_b128(q, ry, vo, 0, 0);
      } else {
        const TOut h0 = from_f32<TOut>(v.x), h1 = from_f32<TOut>(v.y), h2 = from_f32<TOut>(v.z), h3 = from_f32<TOut>(v.w);
        const sf_u32x2 q = {(uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16),
                            (uint32_t)__builtin_bit_cast(uint16_t, h2) | ((uint32_t)__builtin_bit_cast(uint16_t, h3) << 16)};
        __builtin_amdgcn_raw_buffer_store_b64(q, ry, vo, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// One workgroup per 256 x 128 tile (placed XCD-locally: the column blocks
// of a row block run on one XCD and share its rows' words through L2).
template <typename TIn, typename TOut>
__global__ __launch_bounds__(64 * kLbWaves, 2) void k_linear_bits_mfma(LinMfmaArgs a, const uint32_t* __restrict__ bits,
                                                                    const uint32_t* __restrict__ flags, int cwp) {
  __shared__ __align__(16) uint16_t s_wh[kLbBufs][kLmCols * kLmLda];
  __shared__ __align__(16) uint16_t s_wl[kLbBufs][kLmCols * kLmLda];
  __shared__ __align__(16) uint32_t s_words[kLbBufs][kLbRows];  // bitmap word of each row, per step
  __shared__ __align__(16) float s_out[kLbWaves * 16 * 68];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int g = lane >> 4, li = lane & 15;
  const int ncb = (a.c_out + kLmCols - 1) / kLmCols;
  const int nsteps = a.kp / kLmK;
  const int64_t nchunks = (a.m + kLinearRowChunk - 1) / kLinearRowChunk;
  const int bid = xcd_range_block((int)blockIdx.x, (int)gridDim.x);
  const int64_t rb = bid / ncb;
  const int64_t r0 = rb * kLbRows;
  const int c0 = (int)(bid - rb * ncb) * kLmCols;
  const TIn* __restrict__ X = static_cast<const TIn*>(a.x);

  // Step t's bitmap words for the tile's 256 rows (wavefront w: LDS
  // positions 64 w .. 64 w + 63, one word per lane).  Position q holds tile
  // row 128 (q >> 7) + 16 (q & 7) + ((q >> 3) & 15): the words of a lane's
  // eight row tiles (lane li of wavefront row wr: rows 128 wr + 16 rt + li)
  // are consecutive, two 16-byte reads.  Rows past m load row 0's word:
  // their outputs are never stored.
  auto load_step = [&](int t) {
    const int b = t % kLbBufs;
    lb_load_w(s_wh[b], s_wl[b], a.wh, a.wl, a.kp, c0, a.c_out, t, wave, lane);
    const int q = 64 * wave + lane;
    const int64_t row = r0 + 128 * (q >> 7) + 16 * (q & 7) + ((q >> 3) & 15);
    const uint32_t* src = bits + (row < a.m ? row : 0) * (int64_t)cwp + t;
    lds_dma4(src, &s_words[b][64 * wave]);
  };
  auto bfrags = [&](int b, bf16x8 (&bh)[4], bf16x8 (&bl)[4]) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int r = 64 * wc + 16 * ct + li;
      const int c = r * kLmLda + 8 * lm_piece(r, g);
      bh[ct] = *reinterpret_cast<const bf16x8*>(&s_wh[b][c]);
      bl[ct] = *reinterpret_cast<const bf16x8*>(&s_wl[b][c]);
    }
  };
  // Every global load of the spike path is a direct LDS load, waited for by
  // count (the compiler would wait for all of them before the first use of
  // any register load): steps 0 and 1 first, step 0's are waited for.
  load_step(0);
  if (nsteps > 1) load_step(1);
  if (nsteps > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLbLoads) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // The row block's non-binary flags (one per 16 rows, read by every
  // wavefront with uniform loads) decide its A operand.
  uint32_t fl = 0u;
  const int64_t ch0 = r0 / kLinearRowChunk;
#pragma unroll
  for (int i = 0; i < kLbRows / kLinearRowChunk; ++i)
    if (ch0 + i < nchunks) fl |= flags[ch0 + i];
  const bool value = fl != 0u;
  ws_barrier();  // step 0's tiles of every wavefront

  f32x4 acc[kLbRT][4];
#pragma unroll
  for (int i = 0; i < kLbRT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (!value) {
    for (int s = 0; s < nsteps; ++s) {
      const int b = s % kLbBufs;
      // A fragments: byte g of each row tile's word, its 8 bits turned into
      // bf16 0 / 1 on the VALU; B fragments from the W tiles.
      const uint4 w0 = *reinterpret_cast<const uint4*>(&s_words[b][8 * (16 * wr + li)]);
      const uint4 w1 = *reinterpret_cast<const uint4*>(&s_words[b][8 * (16 * wr + li) + 4]);
      const uint32_t wd[kLbRT] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      bf16x8 af[kLbRT];
#pragma unroll
      for (int rt = 0; rt < kLbRT; ++rt) af[rt] = spike_bf16x8(__builtin_amdgcn_ubfe(wd[rt], 8 * g, 8));
      bf16x8 bh[4], bl[4];
      bfrags(b, bh, bl);
#pragma unroll
      for (int rt = 0; rt < kLbRT; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[rt], bh[ct], acc[rt][ct], 0, 0, 0);
#pragma unroll
      for (int rt = 0; rt < kLbRT; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[rt], bl[ct], acc[rt][ct], 0, 0, 0);
      // Step s + 2's loads, behind the MFMAs (its buffer was last read by
      // step s - 1, before the previous barrier); then step s + 1's have
      // landed (only the ones just issued may still be in flight).
      if (s + 2 < nsteps) {
        load_step(s + 2);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLbLoads) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      ws_barrier();
    }
  } else {
    // x tiles: lane (li, g) reads k = 32 s + 8 g .. + 7 of its rows; past k
    // and past m the elements are 0; |x| < cutoff counts as 0.  The eight
    // row tiles in two halves (registers).
    const bool vec4 = sizeof(TIn) == 4 && (a.k & 3) == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0;
    for (int s = 0; s < nsteps; ++s) {
      if (s + 2 < nsteps) load_step(s + 2);  // its buffer was last read by step s - 1
      bf16x8 bh[4], bl[4];
      bfrags(s % kLbBufs, bh, bl);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
      bf16x8 ah[4], al[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const int64_t row = r0 + 128 * wr + 16 * (4 * half + rt) + li;
        const int kk0 = 32 * s + 8 * g;
        float v8[8];
        if (vec4) {
          // f32 rows, k % 4 == 0, 16-byte aligned: two 16-byte loads, each
          // wholly inside or past the row.
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const bool ok = row < a.m && kk0 + 4 * h < a.k;
            const float4 t = *reinterpret_cast<const float4*>(ok ? reinterpret_cast<const float*>(X) + row * a.k + kk0 + 4 * h
                                                                 : reinterpret_cast<const float*>(X));
            v8[4 * h] = ok ? t.x : 0.f;
            v8[4 * h + 1] = ok ? t.y : 0.f;
            v8[4 * h + 2] = ok ? t.z : 0.f;
            v8[4 * h + 3] = ok ? t.w : 0.f;
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int kk = kk0 + e;
            v8[e] = (row < a.m && kk < a.k) ? to_f32<TIn>(X[row * a.k + kk]) : 0.f;
          }
        }
        uint32_t hx[4], lx[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float v2[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) v2[e] = fabsf(v8[2 * j + e]) >= a.cutoff ? v8[2 * j + e] : 0.f;
          const uint16_t h0 = bf16_bits(v2[0]), h1 = bf16_bits(v2[1]);
          hx[j] = (uint32_t)h0 | ((uint32_t)h1 << 16);
          lx[j] = (uint32_t)bf16_bits(v2[0] - bf16_value(h0)) | ((uint32_t)bf16_bits(v2[1] - bf16_value(h1)) << 16);
        }
        ah[rt] = __builtin_bit_cast(bf16x8, make_uint4(hx[0], hx[1], hx[2], hx[3]));
        al[rt] = __builtin_bit_cast(bf16x8, make_uint4(lx[0], lx[1], lx[2], lx[3]));
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          f32x4& c = acc[4 * half + rt][ct];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[rt], bh[ct], c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[rt], bl[ct], c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[rt], bh[ct], c, 0, 0, 0);
        }
      }
      lds_dma_wait();  // the tiles of step s + 1: the compiler does not count them
      __syncthreads();
    }
  }
  // The last step's barrier: every wavefront is done with the buffers.
  const auto rs_y = buf_rsrc(a.y, (uint32_t)((uint64_t)a.m * (uint64_t)a.c_out * sizeof(TOut)));
  lb_store_tile<kLbRT, TOut>(acc, &s_out[wave * 16 * 68], a.bias, rs_y, a.m, a.c_out, r0 + 128 * wr, c0 + 64 * wc,
                             lane);
}

// ---- wide tiles: x staged once for 384 output columns ---------------------
//
// k_linear_mfma's 128 x 128 tiles read (and convert) x once per 128 columns
// and spend a step's time on staging: 32 MFMAs per wavefront between two
// barriers.  Here a workgroup of 8 wavefronts computes 16 RT rows x 384
// columns, each wavefront all rows of 48 columns (RT x 3 MFMA tiles, 6 RT
// MFMAs a step): x is read, tested and converted once for all of them.  x
// goes global -> registers (three steps ahead) -> bf16 in LDS (two steps
// ahead, the conversion between the MFMAs), through four LDS buffers, so
// that one barrier serves two steps; W's hi and lo tiles come by direct loads
// into the other of two buffers and need no barrier, since a wavefront reads
// only the columns it has loaded itself.  A second walk (x's lo part times
// W hi) only where a workgroup saw an element that is not exact in bf16, as
// in k_linear_mfma; same sums in the same order as there.
// Bound by the matrix cores at the rate they hold under load: 50176 x 1536 ->
// 384 runs in 121-127 us, 0.93-0.98 PFLOP/s counting both products (a plain
// bf16 8192^3 product reaches 1.2 here); 191-212 us with k_linear_mfma.
// With x staged one step ahead through two buffers and a barrier per step:
// 125.7; all of a step's staging before its MFMAs, or half of it after them:
// 131, 134.6.
constexpr int kLwWaves = 8;
constexpr int kLwCT = 3;                             // 16-column tiles per wavefront
constexpr int kLwCols = 16 * kLwCT * kLwWaves;       // 384 columns per workgroup
constexpr int kLwWBytes = kLwCols * kLmLda * 2;      // one part of a step's W tiles
constexpr int kLwXBufs = 4;
template <int RT> constexpr int lw_xbytes() { return 16 * RT * kLmLda * 2; }
template <int RT> constexpr int lw_lds() { return 4 * kLwWBytes + kLwXBufs * lw_xbytes<RT>(); }

typedef unsigned int lw_u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane from the raw buffer rs at byte vo + so to LDS byte
// address lds + 16 * lane.  In asm: the compiler would make every later LDS
// read wait for every direct load in flight.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 in the clobber list
__device__ __forceinline__ void lw_load_lds(lw_u32x4 rs, int vo, int so, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(vo), "s"(rs), "s"(so),
               "s"(lds)
               : "m0", "memory");
}
#pragma clang diagnostic pop

__device__ __forceinline__ lw_u32x4 lw_rsrc(const void* p, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(p);
  return lw_u32x4{(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, bytes, 0x00020000u};
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t lw_bf16x2(float v0, float v1) {  // round to nearest even, low half = v0
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v0, v1}, bf16x2));
}

template <typename TIn, typename TOut, int RT, bool VEC>
__global__ __launch_bounds__(64 * kLwWaves, 2) void k_linear_wide(LinMfmaArgs a) {
  extern __shared__ __align__(16) char smem[];
  constexpr int M = 16 * RT;
  constexpr int NX = (M + 63) / 64;  // x loads per thread and step: 64 rows x 8 pieces of four elements each
  constexpr int kXb = lw_xbytes<RT>();
  char* const s_x = smem + 4 * kLwWBytes;  // after two buffers of W's hi and lo tiles
  // VEC: k a multiple of four, x on whole pieces; otherwise rows start anywhere.
  struct __attribute__((packed, aligned((VEC ? 4 : 1) * sizeof(TIn)))) X4 { TIn e[4]; };
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ncb = (a.c_out + kLwCols - 1) / kLwCols;
  const int bid = xcd_range_block((int)blockIdx.x, (int)gridDim.x);
  const int64_t rb = bid / ncb;
  const int64_t r0 = rb * M;
  const int c0 = (int)(bid - rb * ncb) * kLwCols;
  const int nsteps = a.kp / kLmK;
  const TIn* __restrict__ X = static_cast<const TIn*>(a.x);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

  // x: thread t takes rows t / 8 + 64 j, elements 4 (t % 8) .. + 3 of the
  // step.  Rows past m read the last one (their outputs are not stored).
  const int xr = (int)threadIdx.x >> 3, xp = (int)threadIdx.x & 7;
  X4 xv[NX];
  auto load_piece = [&](int s, int j) {
    const int kk = s * kLmK + 4 * xp;
    int64_t row = r0 + min(xr + 64 * j, M - 1);
    row = row < a.m ? row : a.m - 1;
    const TIn* p = X + row * a.k;
    if (VEC || s * kLmK + kLmK <= a.k) {
      xv[j] = *reinterpret_cast<const X4*>(p + (VEC ? min(kk, a.k - 4) : kk));  // (not staged where kk >= k)
    } else {  // the last step of a ragged k: element by element, 0 past the row's end
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[j].e[e] = kk + e < a.k ? p[kk + e] : from_f32<TIn>(0.f);
    }
  };
  uint32_t inexact = 0u;  // some bit set: an element whose lo part is not zero
  auto stage_piece = [&](int s, int j, auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    char* xb = s_x + (s % kLwXBufs) * kXb;
    const bool in = !VEC || s * kLmK + 4 * xp < a.k;
    {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = to_f32<TIn>(xv[j].e[e]);
        v[e] = in && fabsf(v[e]) >= a.cutoff ? v[e] : 0.f;  // the prescan's activity test
      }
      uint32_t h0 = lw_bf16x2(v[0], v[1]), h1 = lw_bf16x2(v[2], v[3]);
      const float l0 = v[0] - __uint_as_float(h0 << 16), l1 = v[1] - __uint_as_float(h0 & 0xffff0000u);
      const float l2 = v[2] - __uint_as_float(h1 << 16), l3 = v[3] - __uint_as_float(h1 & 0xffff0000u);
      if constexpr (LO) {
        h0 = lw_bf16x2(l0, l1);
        h1 = lw_bf16x2(l2, l3);
      } else {
        inexact |= (__float_as_uint(l0) | __float_as_uint(l1) | __float_as_uint(l2) | __float_as_uint(l3)) & 0x7fffffffu;
      }
      const int r = xr + 64 * j;
      if (64 * (j + 1) <= M || r < M)
        *reinterpret_cast<uint2*>(xb + r * (2 * kLmLda) + 16 * lm_piece(r, xp >> 1) + 8 * (xp & 1)) = make_uint2(h0, h1);
    }
  };
  // W: unit u (1 KB) of a part holds columns 16 u .. 16 u + 15 of the tile;
  // LDS position q of a unit holds column q >> 2, stored piece q & 3
  // (lm_piece is its own inverse).  Columns past c_out read column 0 (never
  // stored).  Wavefront w loads units 3 w .. 3 w + 2: its own columns.
  const lw_u32x4 rs_h = lw_rsrc(a.wh, (uint32_t)((int64_t)a.c_out * a.kp * 2));
  const lw_u32x4 rs_l = lw_rsrc(a.wl, (uint32_t)((int64_t)a.c_out * a.kp * 2));
  int wvo[kLwCT];
#pragma unroll
  for (int j = 0; j < kLwCT; ++j) {
    const int r = lane >> 2;
    const int col = c0 + 16 * (kLwCT * wave + j) + r;
    wvo[j] = ((col < a.c_out ? col : 0) * a.kp + 8 * lm_piece(r, lane & 3)) * 2;
  }
  auto load_w = [&](int s, auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    const uint32_t b = lds0 + (uint32_t)((s & 1) * (2 * kLwWBytes));
#pragma unroll
    for (int j = 0; j < kLwCT; ++j) {
      lw_load_lds(rs_h, wvo[j], s * (kLmK * 2), b + (uint32_t)(kLwCT * wave + j) * 1024u);
      if constexpr (!LO) lw_load_lds(rs_l, wvo[j], s * (kLmK * 2), b + kLwWBytes + (uint32_t)(kLwCT * wave + j) * 1024u);
    }
  };

  const int g = lane >> 4, li = lane & 15;
  // MFMA operands W, x: register i of tile (rt, ct) is row 16 rt + li, column
  // 16 ct + 4 g + i of the wavefront's 48: four consecutive columns a lane,
  // stored without an exchange.
  f32x4 acc[RT][kLwCT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < kLwCT; ++ct) acc[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto walk = [&](auto lo_walk) {
    constexpr bool LO = decltype(lo_walk)::value;
    load_w(0, lo_walk);
#pragma unroll
    for (int j = 0; j < NX; ++j) load_piece(0, j);
#pragma unroll
    for (int j = 0; j < NX; ++j) stage_piece(0, j, lo_walk);
    if (nsteps > 1) {
#pragma unroll
      for (int j = 0; j < NX; ++j) load_piece(1, j);
#pragma unroll
      for (int j = 0; j < NX; ++j) stage_piece(1, j, lo_walk);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) load_piece(min(2, nsteps - 1), j);
    ws_barrier();
    for (int s = 0; s < nsteps; ++s) {
      // This wavefront's W tiles of step s and its x of step s + 2, both
      // requested a step ago, have landed (the x is used from here on, so
      // that the compiler's own wait comes before the next direct loads).
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        typedef unsigned int u32xn __attribute__((ext_vector_type(sizeof(X4) / 4)));
        u32xn q = __builtin_bit_cast(u32xn, xv[j]);
        asm volatile("" : "+v"(q));
        xv[j] = __builtin_bit_cast(X4, q);
      }
      if (s + 1 < nsteps) load_w(s + 1, lo_walk);
      const bool more = s + 2 < nsteps;
      const char* buf = smem + (s & 1) * (2 * kLwWBytes);
      const char* xbuf = s_x + (s % kLwXBufs) * kXb;
      bf16x8 bh[kLwCT], bl[kLwCT];
#pragma unroll
      for (int ct = 0; ct < kLwCT; ++ct) {
        const int r = 16 * (kLwCT * wave + ct) + li;
        const char* p = buf + r * (2 * kLmLda) + 16 * lm_piece(r, g);
        bh[ct] = *reinterpret_cast<const bf16x8*>(p);
        if constexpr (!LO) bl[ct] = *reinterpret_cast<const bf16x8*>(p + kLwWBytes);
      }
      auto read_x = [&](int rt) {
        const int r = 16 * rt + li;
        return *reinterpret_cast<const bf16x8*>(xbuf + r * (2 * kLmLda) + 16 * lm_piece(r, g));
      };
      bf16x8 ax = read_x(0);
      // The step's row tiles, the next one's fragment requested ahead; the x
      // of two steps on is converted and stored a piece at a time between them
      // (and the one after it requested), so that it runs beside the MFMAs.
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const bf16x8 an = read_x(rt + 1 < RT ? rt + 1 : rt);
#pragma unroll
        for (int ct = 0; ct < kLwCT; ++ct)
          acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[ct], ax, acc[rt][ct], 0, 0, 0);
        if constexpr (!LO) {
#pragma unroll
          for (int ct = 0; ct < kLwCT; ++ct)
            acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[ct], ax, acc[rt][ct], 0, 0, 0);
        }
        ax = an;
#pragma unroll
        for (int j = 0; j < NX; ++j)
          if (rt == (j * RT) / NX) {
            if (more) {
              stage_piece(s + 2, j, lo_walk);
              load_piece(min(s + 3, nsteps - 1), j);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      // Steps 2 i and 2 i + 1 read two of the x buffers and write the other
      // two: one barrier for both.
      if (s & 1) ws_barrier();
    }
    ws_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  walk(std::false_type{});
  if (__syncthreads_or(inexact != 0u ? 1 : 0)) walk(std::true_type{});

  TOut* __restrict__ Y = static_cast<TOut*>(a.y);
#pragma unroll
  for (int ct = 0; ct < kLwCT; ++ct) {
    const int col = c0 + 16 * (kLwCT * wave + ct) + 4 * g;
    if (col >= a.c_out) continue;  // c_out is a multiple of 4
    const f32x4 b = a.bias == nullptr ? f32x4{0.f, 0.f, 0.f, 0.f}
                                      : f32x4{a.bias[col], a.bias[col + 1], a.bias[col + 2], a.bias[col + 3]};
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int64_t row = r0 + 16 * rt + li;
      const f32x4 v = acc[rt][ct] + b;
      if (row < a.m) store4<TOut>(Y + row * a.c_out + col, v[0], v[1], v[2], v[3]);
    }
  }
}

template <typename TIn>
bool lm_vec(const LinMfmaArgs& a) {  // k_linear_mfma's 16-byte loads
  return sizeof(TIn) == 4 && a.k % 16 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0;
}

// What the choice of a kernel looks at.
struct LinShape {
  int64_t m;
  int k, c_out, e;  // e: bytes of an element of x
  bool vec;         // k_linear_mfma's 16-byte loads
  int cus;
};

LinShape lin_shape(int64_t m, int k, int c_out, int in_dtype, const void* x) {
  const bool f32 = in_dtype == SF_F32;
  return {m, k, c_out, f32 ? 4 : 2, f32 && k % 16 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0,
          num_cus()};
}

// Estimated times of the three kernels (us): per K step and workgroup of a CU
// (per round of workgroups for k_linear_wide), and per MB of y and of x.
// Fitted to 7,000 shapes of k 32 to 2048, c_out 16 to 2048 and up to 131,072
// rows, binary x, inputs and outputs changing from call to call; nine in ten
// estimates are within 15% (short k with a wide y is overestimated, by up to
// a half).
double lin_mb(const LinShape& s, int cols) { return 1e-6 * (double)s.m * cols * s.e; }
int64_t lin_blocks(int64_t n, int64_t per) { return (n + per - 1) / per; }
double lin_per_cu(const LinShape& s, int64_t workgroups) { return (double)lin_blocks(workgroups, s.cus); }

double lm_us(const LinShape& s) {
  const double steps = (double)lin_blocks(s.k, kLmK), y = lin_mb(s, s.c_out), x = lin_mb(s, s.k);
  const double n = lin_per_cu(s, lin_blocks(s.m, kLmRows) * lin_blocks(s.c_out, kLmCols)), n3 = std::ceil(n / 3);
  // Single elements loaded from rows of whole 64-byte lines: every lane's in
  // the same place of its line, a quarter slower.
  const bool in_step = s.k * s.e % 64 == 0;
  if (s.vec) return 2.8 + steps * (0.8 * n3 + 0.32 * n) + 0.197 * y + 0.087 * x;
  if (s.e == 4 && in_step) return 4.0 + steps * (0.47 * n3 + 1.8 * n) + 0.167 * y + 0.07 * x;
  if (s.e == 4) return 2.6 + steps * (0.48 * n3 + 1.44 * n) + 0.122 * y + 0.167 * x;
  if (in_step) return 3.9 + steps * (0.7 * n3 + 1.84 * n) + 0.244 * y + 0.053 * x;
  return 2.6 + steps * (0.61 * n3 + 1.32 * n) + 0.158 * y + 0.142 * x;
}

double lw_us(const LinShape& s, int rt) {
  const double steps = (double)lin_blocks(s.k, kLmK), y = lin_mb(s, s.c_out), x = lin_mb(s, s.k);
  const double rounds = lin_per_cu(s, lin_blocks(s.m, 16 * rt) * lin_blocks(s.c_out, kLwCols));
  if (s.e == 4)  // (a store writes 64 bytes of a row: whole lines where the rows of y start on them)
    return 0.6 + rounds * (4.0 + steps * (0.29 + 0.12 * rt)) + (s.c_out % 16 != 0 ? 0.404 : 0.244) * y + 0.06 * x;
  return 0.5 + rounds * (4.3 + steps * (0.21 + 0.138 * rt)) + 0.46 * y + 0.042 * x;
}

double lb_us(const LinShape& s) {  // with the row prescan
  const double steps = (double)lin_blocks(s.k, kLmK), y = lin_mb(s, s.c_out), x = lin_mb(s, s.k);
  const double n = lin_per_cu(s, lin_blocks(s.m, kLbRows) * lin_blocks(s.c_out, kLmCols));
  if (s.vec) return 10.8 + 0.57 * n + steps * (0.58 + 0.62 * n) + 0.128 * y + 0.177 * x;
  if (s.e == 4) return 8.2 + 1.9 * n + steps * (1.03 + 0.65 * n) + 0.085 * y + 0.16 * x;
  return 7.9 + steps * (2.12 + 0.79 * n) + 0.195 * y + 0.78 * x;
}

// The number of 16-row tiles of a k_linear_wide workgroup, or 0 for
// k_linear_mfma.
//
// A K step of a workgroup takes about 0.6 + 0.15 RT us however many run, one
// workgroup a CU: of 4, 8 and 13 row tiles (all the accumulators that fit)
// the one whose rounds of workgroups take least.
//
// 16-bit x and f32 x with a k that is no multiple of 16 or a start off 16
// bytes, where k_linear_mfma loads and converts single elements: from 128
// columns and k 48 on, but past one round of workgroups only with a k of
// whole pieces of four or at least 160 (a ragged k's last step loads single
// elements here too); one round of 4 row tiles, or of a k from 192 on, pays
// at any width.  us, k_linear_mfma -> wide:
//   f16 (bf16 the same)  50176 x 384 -> 384 135 -> 41.7;  8192 x 512 -> 2048
//   146 -> 49.9;  1000 x 128 -> 128 14.5 -> 7.9;  100000 x 128 -> 128 43.1 ->
//   37.4;  50000 x 48 -> 192 19.3 -> 16.2;  50000 x 386 -> 384 104 -> 46.6;
//   701 x 1790 -> 100 112 -> 48.4;  but 50000 x 64 -> 64 13.6 -> 14.5, 100000
//   x 129 -> 128 35.8 -> 43.6
//   f32  50176 x 1535 -> 384 480 -> 128;  1000 x 383 -> 384 26.7 -> 15.4;
//   300 x 50 -> 128 7.6 -> 7.2;  30000 x 161 -> 640 53.7 -> 38.2;  200 x 1001
//   -> 12 62.2 -> 26.6;  3000 x 99 -> 100 10.9 -> 8.0;  30000 x 200 -> 4 16.6 ->
//   13.1;  but 65536 x 129 -> 512 65.2 -> 67.4, 100000 x 129 -> 128 37.3 -> 46.7,
//   30000 x 99 -> 100 12.7 -> 13.8
//
// Other f32 x, binary (x with a lo part gains more: the second walk shares the
// staging):
//   RT 4:  196 x 384 -> 384 16.2 -> 14.6;  1 x 2048 -> 1000 67.4 -> 51.7;
//          12544 x 1536 -> 384 66.9 -> 50.1;  8192 x 512 -> 512 24.7 -> 22.3
//   RT 8:  25088 x 384 -> 384 30.3 -> 26.5;  3136 x 768 -> 3072 55.9 -> 44.0
//   RT 13: 50176 x 384 -> 384 50.7 -> 40.6;  20000 x 512 -> 1920 112 -> 86
// Short K has no steps to hide the first loads and the stores behind (300 x
// 128 -> 384 8.1 -> 8.4, 32000 x 128 -> 384 16.9 -> 17.9): k >= 192.  Columns
// up to the next 384 are computed and dropped: up to half as many again are
// paid back by the latency in one round of 4 row tiles (16384 x 256 -> 256
// 14.9 -> 13.9), not with more (16384 x 512 -> 512 31.7 -> 33.9, 40000 x 384
// -> 256 31.6 -> 34.0): an eighth there (32768 x 1024 -> 1024 175 -> 146).
// Past one round, the rounds at least three quarters full (100352 x 384 ->
// 384, 0.94: 122 -> 87; 75000 x 384 -> 384, 0.71: 64.3 with k_linear_mfma).
//
// And only where the estimates agree, since columns dropped, rows of y off a
// 64-byte line and a short k add up differently from shape to shape: f16
// 56000 x 132 -> 128 19.1 / 26.4, 65536 x 164 -> 128 23.8 / 29.4; f32 60000 x 164
// -> 400 43.0 / 58.9, 65536 x 132 -> 128 22.4 / 30.3, 16384 x 256 -> 1420 52.0 /
// 73.7 (k_linear_mfma / wide).
int lw_row_tiles(const LinShape& s) {
  if ((int64_t)s.c_out * lin_blocks(s.k, kLmK) * kLmK * 2 >= (1ll << 31)) return 0;  // the buffer offsets' range
  const int64_t cb = lin_blocks(s.c_out, kLwCols), cus = s.cus;
  int rt = 0;
  int64_t best = 0, tiles = 0;
  for (const int r : {4, 8, 13}) {
    const int64_t t = lin_blocks(s.m, 16 * r) * cb, cost = lin_blocks(t, cus) * (4 + r);
    if (rt == 0 || cost < best) {
      rt = r;
      best = cost;
      tiles = t;
    }
  }
  bool wide;
  if (!s.vec) {
    wide = tiles <= cus ? (s.c_out >= 128 && s.k >= 48) || rt == 4 || s.k >= 192
                        : s.c_out >= 128 && s.k >= 48 && (s.k % 4 == 0 || s.k >= 160);
  } else if (s.k < 192) {
    wide = false;
  } else if (rt == 4 && tiles <= cus) {
    wide = 2 * cb * kLwCols <= 3 * (int64_t)s.c_out;
  } else {
    wide = 8 * cb * kLwCols <= 9 * (int64_t)s.c_out &&
           (tiles <= cus || 4 * tiles >= 3 * cus * ((tiles + cus - 1) / cus));
  }
  return wide && lw_us(s, rt) < lm_us(s) ? rt : 0;
}

template <typename TIn, typename TOut, int RT, bool VEC>
int launch_lw_t(const LinMfmaArgs& a, hipStream_t stream) {
  constexpr auto kern = k_linear_wide<TIn, TOut, RT, VEC>;
  const int e = set_lds_limit_once<kern>(kMaxLdsBytes - 1024);  // (the block-wide OR takes a little)
  if (e != (int)hipSuccess) return e;
  const int64_t grid = ((a.m + 16 * RT - 1) / (16 * RT)) * ((a.c_out + kLwCols - 1) / kLwCols);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * kLwWaves), (size_t)lw_lds<RT>(), stream, a);
  return (int)hipGetLastError();
}

template <typename TIn, typename TOut, bool VEC>
int launch_lw_v(const LinMfmaArgs& a, int rt, hipStream_t stream) {
  return rt == 4   ? launch_lw_t<TIn, TOut, 4, VEC>(a, stream)
         : rt == 8 ? launch_lw_t<TIn, TOut, 8, VEC>(a, stream)
                   : launch_lw_t<TIn, TOut, 13, VEC>(a, stream);
}

template <typename TIn, typename TOut>
int launch_lw(const LinMfmaArgs& a, int rt, hipStream_t stream) {
  return a.k % 4 == 0 && reinterpret_cast<uintptr_t>(a.x) % (4 * sizeof(TIn)) == 0
             ? launch_lw_v<TIn, TOut, true>(a, rt, stream)
             : launch_lw_v<TIn, TOut, false>(a, rt, stream);
}

template <typename TIn>
int launch_lb_d(const LinMfmaArgs& a, const uint32_t* bits, const uint32_t* flags, int cwp, int out_dtype,
                hipStream_t stream) {
  const int64_t tiles = ((a.m + kLbRows - 1) / kLbRows) * ((a.c_out + kLmCols - 1) / kLmCols);
  if (tiles == 0) return (int)hipSuccess;
  if (out_dtype == SF_F32)
    hipLaunchKernelGGL((k_linear_bits_mfma<TIn, float>), dim3((unsigned)tiles), dim3(64 * kLbWaves), 0, stream, a,
                       bits, flags, cwp);
  else
    hipLaunchKernelGGL((k_linear_bits_mfma<TIn, TIn>), dim3((unsigned)tiles), dim3(64 * kLbWaves), 0, stream, a, bits,
                       flags, cwp);
  return (int)hipGetLastError();
}

template <typename TIn>
int launch_lm_d(const LinMfmaArgs& a, int out_dtype, hipStream_t stream) {
  const int rt = lw_row_tiles(lin_shape(a.m, a.k, a.c_out, sizeof(TIn) == 4 ? SF_F32 : SF_F16, a.x));
  if (rt != 0) return out_dtype == SF_F32 ? launch_lw<TIn, float>(a, rt, stream) : launch_lw<TIn, TIn>(a, rt, stream);
  const int64_t rbs = (a.m + kLmRows - 1) / kLmRows;
  const int64_t grid = rbs * ((a.c_out + kLmCols - 1) / kLmCols);
  if (grid == 0) return (int)hipSuccess;
  if (lm_vec<TIn>(a)) {
    if (out_dtype == SF_F32)
      hipLaunchKernelGGL((k_linear_mfma<TIn, float, true>), dim3((unsigned)grid), dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((k_linear_mfma<TIn, TIn, true>), dim3((unsigned)grid), dim3(256), 0, stream, a);
  } else {
    if (out_dtype == SF_F32)
      hipLaunchKernelGGL((k_linear_mfma<TIn, float, false>), dim3((unsigned)grid), dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((k_linear_mfma<TIn, TIn, false>), dim3((unsigned)grid), dim3(256), 0, stream, a);
  }
  return (int)hipGetLastError();
}

}  // namespace

int linear_mfma_max_kp() { return kLmMaxK; }

int linear_mfma_row_tiles(const void* x, int in_dtype, int64_t m, int k, int c_out) {
  return lw_row_tiles(lin_shape(m, k, c_out, in_dtype, x));
}

// Whether the row prescan and k_linear_bits_mfma beat the direct kernels: from
// outputs twice as wide as the input on, the large ones as measured here and
// the others by the estimates (us, bitmap / direct, 10% spikes):
//   f32   50176 x 384 -> 1536  153 / 165    32768 x 512 -> 2048  146 / 184
//         65536 x 192 -> 768   63 / 71      65536 x 160 -> 1280  92 / 132
//         25088 x 384 -> 1536  81 / 71      8192 x 512 -> 2048   50 / 46
//         4096 x 1024 -> 4096  81 / 73      1000 x 384 -> 1536   29 / 15
//         65536 x 128 -> 512   42 / 36      65536 x 128 -> 1536  93 / 143
//         8192 x 768 -> 3072   98 / 85      10000 x 64 -> 256    16 / 7
//   f16   50176 x 384 -> 1536  158 / 157    8192 x 512 -> 2048   80 / 50
//         65536 x 192 -> 768   72 / 79      8192 x 768 -> 3072   153 / 89
//         65536 x 128 -> 512   42 / 52      32768 x 128 -> 512   31 / 28
//   f32, k no multiple of 16 or x off 16 bytes
//         50176 x 385 -> 1536  172 / 216    58638 x 192 -> 744   71 / 122
//         30000 x 132 -> 772   37 / 49      16384 x 50 -> 820    21 / 24
//         66745 x 68 -> 324    36 / 47      8192 x 128 -> 1716   25 / 39
// (x of full precision is faster direct throughout: 50176 x 384 -> 1536 408 /
// 239.)  On binary x both give the same bits.
bool linear_mfma_bits_pays(const void* x, int in_dtype, int64_t m, int k, int c_out) {
  if (c_out < 2 * k || m * (int64_t)linear_words_per_row(k) * 4 >= (1ll << 31)) return false;
  const LinShape s = lin_shape(m, k, c_out, in_dtype, x);
  if (k < 192 ? !s.vec && m * c_out >= 25000000 : m * c_out >= 45000000) return true;
  // Two launches instead of one: the host needs about 30 us for them.
  const int rt = lw_row_tiles(s);
  return 1.03 * (rt != 0 ? lw_us(s, rt) : lm_us(s)) >= std::max(lb_us(s), 30.0);
}

int launch_linear_bits_mfma(const LinMfmaArgs& a, const uint32_t* bits, const uint32_t* flags, int cwp, int in_dtype,
                            int out_dtype, hipStream_t stream) {
  timing_begin(K_LINEAR_MFMA, stream);
  const int rc = in_dtype == SF_F16    ? launch_lb_d<__half>(a, bits, flags, cwp, out_dtype, stream)
                 : in_dtype == SF_BF16 ? launch_lb_d<__hip_bfloat16>(a, bits, flags, cwp, out_dtype, stream)
                                       : launch_lb_d<float>(a, bits, flags, cwp, out_dtype, stream);
  timing_end(K_LINEAR_MFMA, stream);
  return rc;
}

int launch_linear_mfma(const LinMfmaArgs& a, int in_dtype, int out_dtype, hipStream_t stream) {
  timing_begin(K_LINEAR_MFMA, stream);
  const int rc = in_dtype == SF_F16    ? launch_lm_d<__half>(a, out_dtype, stream)
                 : in_dtype == SF_BF16 ? launch_lm_d<__hip_bfloat16>(a, out_dtype, stream)
                                       : launch_lm_d<float>(a, out_dtype, stream);
  timing_end(K_LINEAR_MFMA, stream);
  return rc;
}

}  // namespace sf
