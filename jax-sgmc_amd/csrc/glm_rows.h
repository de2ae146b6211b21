// Row loop of the GLM kernels: gather of float4 row chunks, row dot products, the
// likelihood and its derivative, gradient accumulation, block reduction.
//
// Row layout in HBM: X is row-major [N, ldx] float32 with ldx a multiple of 4 and
// 16-byte aligned rows; a row is read as float4 chunks, chunk c by lane c % LPR of a
// segment of LPR lanes, so a wavefront covers 64/LPR rows per load instruction and
// every load is a contiguous 16*LPR-byte run. Rows are reduced with xor-shuffles
// inside the segment; the per-lane gradient accumulators are reduced across segments,
// then across the block's wavefronts through LDS, then across blocks by the last
// block to arrive (deterministic order).
#pragma once
#include <math.h>

#include "glm_common.h"
#include "sgmc_common.h"
#include "sgmc_device.h"

namespace sgmc {

constexpr int kNT = 256;
constexpr int kWaves = kNT / kWave;
constexpr int kMaxD = 1024;  // fused path: features per row
constexpr int kLdsRows = 4096;  // per-row likelihoods staged in LDS per block
constexpr int kResWindow = 512;  // resident loop: step sizes / save slots staged per window

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dot4(float4 a, float4 b) {
  return ((a.x * b.x + a.y * b.y) + a.z * b.z) + a.w * b.w;
}

__device__ __forceinline__ float dot4(f4 a, float4 b) {
  return ((a.x * b.x + a.y * b.y) + a.z * b.z) + a.w * b.w;
}

__device__ __forceinline__ void axpy4(float4& acc, float r, float4 x) {
  acc.x += r * x.x;
  acc.y += r * x.y;
  acc.z += r * x.z;
  acc.w += r * x.w;
}

__device__ __forceinline__ void axpy4(float4& acc, float r, f4 x) {
  acc.x += r * x.x;
  acc.y += r * x.y;
  acc.z += r * x.z;
  acc.w += r * x.w;
}

// Source of the row index of minibatch row j.
struct RowSource {
  const int32_t* idx;  // explicit indices, or null
  int draw;            // nonzero: in-kernel randint with (k1, k2)
  Key k1, k2;
  uint32_t n, span, mult, magic;
  int64_t rows;        // rows addressable through X (bounds guard)
  // Row index of minibatch row j, or -1 if it falls outside [0, rows).
  __device__ __forceinline__ int64_t row(int j) const {
    int64_t r;
    if (draw) r = (int64_t)draw_index(k1, k2, n, (uint32_t)j, span, mult, magic);
    else if (idx) r = (int64_t)idx[j];
    else r = (int64_t)j;
    return (r >= 0 && r < rows) ? r : -1;
  }
};

// Sum over the LPR lanes of a segment (segments are aligned runs of LPR lanes); every
// lane of the segment gets the sum. Steps inside a 16-lane row use DPP (quad
// permutes, half-row and row mirrors), the xor-16 step a lane swap, the last step
// two readlanes.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF,
                                                        false));
}

template <int LPR>
__device__ __forceinline__ float seg_sum(float v) {
  if (LPR >= 2) v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
  if (LPR >= 4) v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
  if (LPR >= 8) v = dpp_add<0x141>(v);  // row_half_mirror
  if (LPR >= 16) v = dpp_add<0x140>(v); // row_mirror
  if (LPR >= 32) v = xor16_add(v);
  if (LPR >= 64)
    v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)) +
        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  return v;
}

// Rows in flight per segment per pipeline stage: 4, also for D > 512 (eight 4 KB rows in
// flight per wavefront there; 2 rows per stage left the row loop latency-bound); a stage
// of RPW-row loads never exceeds one 64-row chunk.
template <int LPR, int CPL>
struct Unroll {
  static constexpr int U0 = 4;
  static constexpr int U = U0 < LPR ? U0 : LPR;
};

// Row ids of one 64-row chunk of a wavefront's range: lane l holds the id of row cb + l
// (-1 when outside [0, rows) or past the range end). Labels are loaded with the rows'
// features, so nothing here has to be waited on before the next loads are issued. At
// most 32 drawn rows take their two randint words on the two lane halves (lanes 0-31 the
// words of k1, lanes 32-63 those of k2), one Threefry block of latency instead of two.
// Every lane of the wavefront calls this.
__device__ __forceinline__ int chunk_rows(const RowSource& src, int cb, int r1) {
  const int lane = threadIdx.x & (kWave - 1);
  int rid = -1;
  if (src.draw && r1 - cb <= kWave / 2) {
    const int rr = lane & (kWave / 2 - 1);
    const bool low = lane < kWave / 2;
    const Key kk = {low ? src.k1.k0 : src.k2.k0, low ? src.k1.k1 : src.k2.k1};
    const uint32_t word = bits_word(kk, src.n, (uint32_t)min(cb + rr, r1 - 1));
    uint32_t hi;
    lane_swap32(word, hi);  // the k2 word of row rr
    if (low && cb + rr < r1) {
      const int64_t r = (int64_t)(int32_t)randint_offset(word, hi, src.span, src.mult, src.magic);
      if (r >= 0 && r < src.rows) rid = (int)r;
    }
    return rid;
  }
  if (cb + lane < r1) {
    const int64_t r = src.row(cb + lane);
    if (r >= 0) rid = (int)r;
  }
  return rid;
}

template <int LPR, int CPL>
struct RowGroup {
  static constexpr int U = Unroll<LPR, CPL>::U;
  f4 x[U][CPL];
  float y[U];
  bool ok[U];
};

// Buffer resource word 3 for raw (unformatted) buffer loads on CDNA.
constexpr int kRawBufferFlags = 0x00020000;

// Issues the loads of the U row groups starting at group-local offset gl of a chunk.
// Rows of a whole wavefront (LPR = 64) are read through a buffer resource whose base is
// the row and whose size is the row's 4 D4 floats: the base lives in scalar registers,
// the chunks are one lane offset plus immediate offsets, and chunks past the row (or
// every chunk of a row outside the data, size 0) read as zero without a clamp.
template <int LPR, int CPL>
__device__ __forceinline__ void load_group(gcfloat* __restrict__ X, int64_t ldx,
                                           gcfloat* __restrict__ y, int D4, int gl, int rid,
                                           RowGroup<LPR, CPL>& g) {
  constexpr int RPW = kWave / LPR;
  constexpr int U = RowGroup<LPR, CPL>::U;
  const int lane = threadIdx.x & (kWave - 1);
  const int seg = lane / LPR;
  const int q = lane % LPR;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int sl = gl + u * RPW + seg;  // < 64
    int r;
    if (RPW == 1) r = __builtin_amdgcn_readlane(rid, sl);
    else r = __shfl(rid, sl, kWave);
    g.ok[u] = r >= 0;
    const int64_t rc = r >= 0 ? r : 0;
    g.y[u] = y[rc];
    if constexpr (RPW == 1) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(const float*)(X + rc * ldx), (short)0, r >= 0 ? 16 * D4 : 0, kRawBufferFlags);
#pragma unroll
      for (int k = 0; k < CPL; ++k)
        g.x[u][k] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(
                                               rs, 16 * (q + LPR * k), 0, 0));
    } else {
      SGMC_GLOBAL const f4* rp = reinterpret_cast<SGMC_GLOBAL const f4*>(X + rc * ldx);
      // every lane loads (clamped to a valid chunk); invalid chunks are zeroed at use
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        const int c4 = q + LPR * k;
        g.x[u][k] = rp[c4 < D4 ? c4 : D4 - 1];
      }
    }

  }
}

// Dot product and accumulation of the row loop with fused multiply-adds.
__device__ __forceinline__ float dot4_fma(f4 a, float4 b, float t) {
  t = fmaf(a.x, b.x, t);
  t = fmaf(a.y, b.y, t);
  t = fmaf(a.z, b.z, t);
  return fmaf(a.w, b.w, t);
}

__device__ __forceinline__ void axpy4_fma(float4& acc, float r, f4 x) {
  acc.x = fmaf(r, x.x, acc.x);
  acc.y = fmaf(r, x.y, acc.y);
  acc.z = fmaf(r, x.z, acc.z);
  acc.w = fmaf(r, x.w, acc.w);
}

// One row group: z = x . w per row (segment sums), the likelihood and dlik/dz of row u
// evaluated once, by lane u of the row's segment, and broadcast; then acc += r x.
template <int LPR, int CPL>
__device__ __forceinline__ void process_group(RowGroup<LPR, CPL>& g, int row0, int D4,
                                              const float4 (&th)[CPL], const Lik& L,
                                              float4 (&acc)[CPL], float& lik_acc,
                                              float* lds_lik, int lds_row0) {
  constexpr int RPW = kWave / LPR;
  constexpr int U = RowGroup<LPR, CPL>::U;
  static_assert(U <= LPR, "one lane per row of the group");
  const int lane = threadIdx.x & (kWave - 1);
  const int seg = lane / LPR;
  const int q = lane % LPR;
  // chunks past D (clamped loads) and rows outside the data contribute zero; the
  // masking is skipped when the whole wavefront's group is valid, and always for rows
  // read through a buffer resource (those chunks read as zero)
  bool bad = RPW > 1 && D4 < LPR * CPL;
#pragma unroll
  for (int u = 0; u < U; ++u) bad = bad || (RPW > 1 && !g.ok[u]);
  if (__any(bad)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        const bool valid = g.ok[u] && (q + LPR * k) < D4;
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
        g.x[u][k] = valid ? g.x[u][k] : zero;
      }
    }
  }
  float z[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < CPL; ++k) t = dot4_fma(g.x[u][k], th[k], t);
    z[u] = seg_sum<LPR>(t);
  }
  // lane q < U of each segment takes row q (bitwise blends: a select chain on q would be
  // turned into an indexed table in scratch memory)
  uint32_t zb = __float_as_uint(z[0]), yb = __float_as_uint(g.y[0]);
  uint32_t okb = g.ok[0] ? 1u : 0u;
#pragma unroll
  for (int u = 1; u < U; ++u) {
    const uint32_t m = 0u - (uint32_t)(q == u);
    zb = (zb & ~m) | (__float_as_uint(z[u]) & m);
    yb = (yb & ~m) | (__float_as_uint(g.y[u]) & m);
    okb = (okb & ~m) | ((g.ok[u] ? 1u : 0u) & m);
  }
  const float zq = __uint_as_float(zb), yq = __uint_as_float(yb);
  const bool okq = okb != 0u;
  float likq, rq;
  row_lik(L, zq, yq, likq, rq);
  if (!okq) {
    likq = 0.0f;
    rq = 0.0f;
  }
  if (q < U && okq) {
    lik_acc += likq;
    lds_lik[row0 + q * RPW + seg - lds_row0] = likq;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float r;
    if (RPW == 1) r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rq), u));
    else r = __shfl(rq, seg * LPR + u, kWave);
#pragma unroll
    for (int k = 0; k < CPL; ++k) axpy4_fma(acc[k], r, g.x[u][k]);
  }
}

// Accumulates sum_j r_j x_j (this lane's chunks) and sum_j lik_j over minibatch rows
// [r0, r1). Loads run one row group ahead of the arithmetic (two register buffers), and
// the row ids of the next 64-row chunk are drawn before the current chunk is done. mid()
// runs (on every wavefront, also one without rows) when the first loads are in flight: it
// sets th, and whatever else does not depend on the rows is hidden behind them.
// Where a lane adds every row (D > 128), the float32 sums are kept in two levels, chunks of 64
// rows and their sum: a wavefront of a long block has hundreds of rows (256 at 64 chains of
// n = 4096), and one running sum over them rounds more than the many short blocks of a finer
// split did. Errors of SGHMC of 64 chains, n = 4096, against 64 bits, one sum and two levels:
// D = 200 2.6e-7 2.5e-7, D = 512 2.9e-7 2.6e-7, D = 900 2.5e-7 2.4e-7, at the same times within
// 0.5%; D = 60 and 100, several rows per load, 3.9e-7 and 5.0e-7 either way (and 1% slower).
template <int LPR, int CPL, class Mid>
__device__ __forceinline__ void accumulate_rows(gcfloat* __restrict__ X, int64_t ldx,
                                                gcfloat* __restrict__ y, int D4,
                                                const RowSource& src, int r0, int r1,
                                                const float4 (&th)[CPL], const Lik& L,
                                                float4 (&acc)[CPL], float& lik_acc,
                                                float* lds_lik, int lds_row0, Mid mid) {
  constexpr int RPW = kWave / LPR;
  constexpr int G = RPW * RowGroup<LPR, CPL>::U;  // rows per group; divides 64
  constexpr bool kTwo = RPW == 1;  // sums in two levels
  static_assert(kWave % G == 0, "row groups must tile a 64-row chunk");
  if (r0 >= r1) {
    mid();
    return;
  }
  int cb = r0;
  int rid = chunk_rows(src, cb, r1);
  RowGroup<LPR, CPL> ga, gb;
  float4 tot[CPL];
  float lik_tot = 0.0f;
#pragma unroll
  for (int k = 0; k < CPL; ++k) tot[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  auto fold = [&] {
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
      tot[k] = make_float4(tot[k].x + acc[k].x, tot[k].y + acc[k].y, tot[k].z + acc[k].z,
                           tot[k].w + acc[k].w);
      acc[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    lik_tot += lik_acc;
    lik_acc = 0.0f;
  };
  load_group<LPR, CPL>(X, ldx, y, D4, 0, rid, ga);
  int rid_n = cb + kWave < r1 ? chunk_rows(src, cb + kWave, r1) : -1;
  mid();
  int gl = 0;  // group offset inside the current chunk
  // The prefetch is issued on every path (rows past the range carry id -1 and load the
  // clamped row 0), so the number of loads in flight is the same on every path and the
  // wait before the arithmetic only covers the group being processed.
  for (;;) {
    int nl = gl + G;
    bool more = cb + nl < r1;
    bool next = nl >= kWave;
    load_group<LPR, CPL>(X, ldx, y, D4, next ? 0 : nl, next ? rid_n : rid, gb);
    process_group<LPR, CPL>(ga, cb + gl, D4, th, L, acc, lik_acc, lds_lik, lds_row0);
    if (!more) break;
    if (next) {
      if (kTwo) fold();
      cb += kWave;
      nl = 0;
      rid = rid_n;
      rid_n = cb + kWave < r1 ? chunk_rows(src, cb + kWave, r1) : -1;
    }
    gl = nl;
    nl = gl + G;
    more = cb + nl < r1;
    next = nl >= kWave;
    load_group<LPR, CPL>(X, ldx, y, D4, next ? 0 : nl, next ? rid_n : rid, ga);
    process_group<LPR, CPL>(gb, cb + gl, D4, th, L, acc, lik_acc, lds_lik, lds_row0);
    if (!more) break;
    if (next) {
      if (kTwo) fold();
      cb += kWave;
      nl = 0;
      rid = rid_n;
      rid_n = cb + kWave < r1 ? chunk_rows(src, cb + kWave, r1) : -1;
    }
    gl = nl;
  }
  if (kTwo && r1 - r0 > kWave) {
    fold();
#pragma unroll
    for (int k = 0; k < CPL; ++k) acc[k] = tot[k];
    lik_acc = lik_tot;
  }
}

// v + (v of lane l ^ M).
template <int M>
__device__ __forceinline__ float xor_add(float v) {
  if (M == 32) return xor32_add(v);
  if (M == 16) return xor16_add(v);
  if (M == 8) return ror_add<8>(v);
  return v + __shfl_xor(v, M, kWave);
}
template <int M>
__device__ __forceinline__ void xor_add4(float4& a) {
  a = make_float4(xor_add<M>(a.x), xor_add<M>(a.y), xor_add<M>(a.z), xor_add<M>(a.w));
}

// Reduces acc over the segments of each wavefront and leaves the wavefronts' sums in
// lds_cols ([kWaves][4 D4]) and their lik sums in lds_small; returns the block's lik sum.
// One barrier: lds_cols and lds_small must not be in use by a slower wavefront.
template <int LPR, int CPL>
__device__ __forceinline__ float block_reduce(float4 (&acc)[CPL], float lik_acc, int D4,
                                              float* lds_cols, float* lds_small) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int q = lane % LPR;
#pragma unroll
  for (int k = 0; k < CPL; ++k) {
    if (LPR <= 4) xor_add4<4>(acc[k]);
    if (LPR <= 8) xor_add4<8>(acc[k]);
    if (LPR <= 16) xor_add4<16>(acc[k]);
    if (LPR <= 32) xor_add4<32>(acc[k]);
  }
  if (lane < LPR) {
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
      const int c4 = q + LPR * k;
      if (c4 < D4) reinterpret_cast<float4*>(lds_cols + w * 4 * D4)[c4] = acc[k];
    }
  }
  lik_acc = wave_sum(lik_acc);
  if (lane == 0) lds_small[w] = lik_acc;
  __syncthreads();
  float lsum = 0.0f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) lsum += lds_small[i];
  return lsum;
}

// Column sum c over the wavefronts.
__device__ __forceinline__ float col_sum(const float* lds_cols, int D4, int c) {
  float s = 0.0f;
#pragma unroll
  for (int ww = 0; ww < kWaves; ++ww) s += lds_cols[ww * 4 * D4 + c];
  return s;
}

// Splits rows [0, n) of a minibatch among the blocks of a chain and then among the
// wavefronts of a block (contiguous ranges).
__device__ __forceinline__ void wave_rows(int n, int nblocks, int b, int& r0, int& r1,
                                          int& b0, int& b1) {
  const int per_block = (n + nblocks - 1) / nblocks;
  b0 = min(n, b * per_block);
  b1 = min(n, b0 + per_block);
  const int per_wave = (b1 - b0 + kWaves - 1) / kWaves;
  const int w = threadIdx.x / kWave;
  r0 = min(b1, b0 + w * per_wave);
  r1 = min(b1, r0 + per_wave);
}

template <int LPR, int CPL>
__device__ __forceinline__ void load_theta(gcfloat* w, int D, float4 (&th)[CPL]) {
  const int q = (threadIdx.x & (kWave - 1)) % LPR;
#pragma unroll
  for (int k = 0; k < CPL; ++k) {
    const int c = 4 * (q + LPR * k);
    th[k].x = c + 0 < D ? w[c + 0] : 0.f;
    th[k].y = c + 1 < D ? w[c + 1] : 0.f;
    th[k].z = c + 2 < D ? w[c + 2] : 0.f;
    th[k].w = c + 3 < D ? w[c + 3] : 0.f;
  }
}

}  // namespace sgmc
