// Full-data potential of many chains at once (potential.py:219-293 for every chain of
// a table that shares one dataset): U_c = (-sum_i lik(x_i . theta_c, y_i) - log p(theta_c))
// / T, each chain's sum over rows accumulated in FP64.
//
// The row dot products for all chains form the product Z = X Theta^T of the [N, D] rows
// and the [C, D] positions, so they run on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32) and X is read from HBM once for up to 64 chains instead of
// once per chain. Layout:
// - Theta^T is staged once per block in LDS in B-operand order: for k-block j (eight
//   columns), chain tile t (32 chains) and lane l, the float4
//   Theta[32 t + l % 32][8 j + 4 (l / 32) + 0..3] (128 KiB at D = 512 and 64 chains);
// - each wave takes 64-row tiles (two 32-row groups); lane l streams the float4
//   x[row + l % 32][8 j + 4 (l / 32) + 0..3] straight from HBM into the A operand, four
//   k-blocks ahead of the matrix instructions. Within the eight columns of a k-block
//   the lane halves split the sum as the two K entries of the instruction, so the sum
//   over columns runs in a fixed, permuted order;
// - the 32x32 accumulator of (row group, chain tile) holds z[m][n] at register r of
//   lane l with n = l % 32, m = 8 (r / 4) + 4 (l / 32) + r % 4; the likelihood is
//   applied there and summed per chain in FP64, then across lanes, waves and blocks
//   (blocks in order by the last block to arrive), so the result is deterministic.
#include <math.h>

#include <type_traits>

#include "glm_common.h"
#include "sgmc_common.h"
#include "sgmc_device.h"

namespace sgmc {
namespace {

constexpr int kFcThreads = 512;
constexpr int kFcWaves = kFcThreads / kWave;
constexpr int kFcLdsF4 = 8192;     // float4 entries of Theta operands (128 KiB)
constexpr int kFcAhead = 4;        // k-blocks of A loads in flight per row group
constexpr int kFcChainsMax = 64;

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

struct FcArgs {
  const float* X;
  const float* y;
  const float* thetas;   // chain c at thetas + c * ld_theta
  double* out_U;         // [nchains]
  double* partial;       // [gridDim.x][kFcChainsMax]
  unsigned* counter;
  int64_t ldx;
  int64_t ld_theta;
  int64_t N;
  int64_t tiles;         // ceil(N / 64), split kernel: ceil(N / kTile)
  int D;
  int D4;                // ceil(D / 4): float4 columns of a row that may be read
  int D8r;               // ceil(D / 8) rounded up to kFcAhead
  int nchains;           // chains of this launch (<= 32 NT)
  int x_exp;             // split kernel: X is scaled by 2^x_exp before splitting
  Lik L;
  Prior pr;
  double temperature;
};

// Branch-free: the load always goes to a valid address (column 0 of a valid row when
// out of range) and the value is masked afterwards, so the loads stay in flight across
// loop iterations instead of being drained at every branch.
__device__ __forceinline__ v4f load_x4(const float* row, int c4, bool ok, int D4) {
  const bool in = ok && c4 < D4;
  const v4f v = *reinterpret_cast<const v4f*>(row + 4 * (in ? c4 : 0));
  const v4f z = {0.f, 0.f, 0.f, 0.f};
  return in ? v : z;
}

// The products of k-blocks jb .. jb + kFcAhead - 1 for both row groups and all chain
// tiles, A operands in registers and B operands from LDS.
template <int NT>
__device__ __forceinline__ void mma_group(v16f (&acc)[2][NT], const v4f (&cur0)[kFcAhead],
                                          const v4f (&cur1)[kFcAhead], const v4f* lds_b,
                                          int jb, int lane) {
  v4f b[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) b[t] = lds_b[(jb * NT + t) * kWave + lane];
#pragma unroll
  for (int u = 0; u < kFcAhead; ++u) {
    // B operands of the next k-block are read while this one's products run.
    v4f bn[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
      bn[t] = u + 1 < kFcAhead ? lds_b[((jb + u + 1) * NT + t) * kWave + lane] : b[t];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        acc[0][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur0[u][tt], b[t][tt], acc[0][t], 0, 0,
                                                         0);
        acc[1][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur1[u][tt], b[t][tt], acc[1][t], 0, 0,
                                                         0);
      }
#pragma unroll
    for (int t = 0; t < NT; ++t) b[t] = bn[t];
  }
}

// Per-row likelihood of one family. The logistic softplus uses the hardware base-2
// exponential and logarithm (about 1 ulp each): log(1 + e^-|z|) = ln2 log2(1 + 2^(-|z|
// log2 e)); where 1 + e^-|z| rounds to 1 the dropped term is below 2^-24, so each row
// is within a few float32 ulps of the exact value while costing a tenth of the
// library routines.
template <int FAM>
__device__ __forceinline__ float fam_lik(const Lik& L, float z, float y) {
  if (FAM == SGMC_LIK_LINEAR_GAUSSIAN) {
    const float d = y - z;
    return (L.log_norm + (d * d) * L.inv_s2) / -2.0f;
  }
  constexpr float kLog2e = 1.44269504088896340736f;
  constexpr float kLn2 = 0.69314718055994530942f;
  const float e = __builtin_amdgcn_exp2f(-fabsf(z) * kLog2e);
  const float sp = fmaxf(z, 0.0f) + __builtin_amdgcn_logf(1.0f + e) * kLn2;
  return y * z - sp;
}

// The last block: sums every chain's block records and forms U. Eight threads per chain
// (64 chains of 512 threads) take every eighth block and prior term, then the eight sums are
// added in order.
__device__ __forceinline__ void finish_chains(const FcArgs& a, double (*red)[kFcChainsMax]) {
  const int c = threadIdx.x % kFcChainsMax, sub = threadIdx.x / kFcChainsMax;
  double tot = 0.0, lp = 0.0;
  if (c < a.nchains) {
    // sixteen records per memory round trip (missing ones add +0)
    for (int b0 = sub; b0 < (int)gridDim.x; b0 += 16 * kFcWaves) {
      double v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int b = b0 + i * kFcWaves;
        v[i] = consume(a.partial + (int64_t)min(b, (int)gridDim.x - 1) * kFcChainsMax + c);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) tot += b0 + i * kFcWaves < (int)gridDim.x ? v[i] : 0.0;
    }
    if (a.pr.has_prior) {
      const double iv = (double)a.pr.inv_var;
      const double ln = (double)a.pr.log_norm;
      const float* th = a.thetas + (int64_t)c * a.ld_theta;
#pragma unroll 8
      for (int k = sub; k < a.D; k += kFcWaves) {
        const double wk = (double)th[k];
        lp += (ln + wk * wk * iv) / -2.0;
      }
    }
  }
  __syncthreads();
  red[sub][c] = -tot - lp;
  __syncthreads();
  if (threadIdx.x >= a.nchains) return;
  double u = 0.0;
  for (int v = 0; v < kFcWaves; ++v) u += red[v][threadIdx.x];
  a.out_U[threadIdx.x] = u / a.temperature;
}

template <int NT, int FAM>
__global__ void __launch_bounds__(kFcThreads) glm_full_chains_kernel(FcArgs a) {
  __shared__ v4f lds_b[kFcLdsF4];
  __shared__ double lds_red[kFcWaves][kFcChainsMax];
  __shared__ int flag;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int rsub = lane & 31;
  const int q = lane >> 5;

  // Theta operands: entry e = (j * NT + t) * 64 + l. Every load of the thread is
  // issued before the first LDS store (clamped addresses, masked values).
  const int entries = a.D8r * NT * kWave;
  constexpr int kPer = kFcLdsF4 / kFcThreads;
  v4f stage[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = threadIdx.x + i * kFcThreads;
    const int l = e % kWave;
    const int t = (e / kWave) % NT;
    const int j = e / (kWave * NT);
    const int c = 32 * t + (l & 31);
    const int k0 = 8 * j + 4 * (l >> 5);
    const bool live = e < entries && c < a.nchains;
    const float* src = a.thetas + (int64_t)(live ? c : 0) * a.ld_theta;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool ok = live && k0 + u < a.D;
      const float x = src[ok ? k0 + u : 0];
      v[u] = ok ? x : 0.0f;
    }
    stage[i] = v4f{v[0], v[1], v[2], v[3]};
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = threadIdx.x + i * kFcThreads;
    if (e < entries) lds_b[e] = stage[i];
  }
  __syncthreads();

  const int64_t t0 = (int64_t)blockIdx.x * a.tiles / gridDim.x;
  const int64_t t1 = (int64_t)(blockIdx.x + 1) * a.tiles / gridDim.x;
  double sacc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) sacc[t] = 0.0;

  for (int64_t tile = t0 + w; tile < t1; tile += kFcWaves) {
    const int64_t r0 = tile * 64 + rsub;
    const int64_t r1 = r0 + 32;
    const bool ok0 = r0 < a.N, ok1 = r1 < a.N;
    const float* x0 = a.X + (ok0 ? r0 : 0) * a.ldx;
    const float* x1 = a.X + (ok1 ? r1 : 0) * a.ldx;
    v16f acc[2][NT];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[g][t] = v16f{};
    v4f cur0[kFcAhead], cur1[kFcAhead];
#pragma unroll
    for (int u = 0; u < kFcAhead; ++u) {
      cur0[u] = load_x4(x0, 2 * u + q, ok0, a.D4);
      cur1[u] = load_x4(x1, 2 * u + q, ok1, a.D4);
    }
    const int jlast = a.D8r - kFcAhead;
    for (int jb = 0; jb < jlast; jb += kFcAhead) {
      v4f nxt0[kFcAhead], nxt1[kFcAhead];
#pragma unroll
      for (int u = 0; u < kFcAhead; ++u) {
        const int c4 = 2 * (jb + kFcAhead + u) + q;
        nxt0[u] = load_x4(x0, c4, ok0, a.D4);
        nxt1[u] = load_x4(x1, c4, ok1, a.D4);
      }
      mma_group<NT>(acc, cur0, cur1, lds_b, jb, lane);
#pragma unroll
      for (int u = 0; u < kFcAhead; ++u) {
        cur0[u] = nxt0[u];
        cur1[u] = nxt1[u];
      }
    }
    // Labels of the lane's 32 accumulator rows, loaded while the last k-blocks run
    // (clamped index, masked below).
    float yv[2][16];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = tile * 64 + 32 * g + 8 * (r / 4) + 4 * q + (r % 4);
        yv[g][r] = a.y[row < a.N ? row : a.N - 1];
      }
    mma_group<NT>(acc, cur0, cur1, lds_b, jlast, lane);
    // Likelihood of every (row, chain) entry of the tile, summed per chain in FP64.
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = tile * 64 + 32 * g + 8 * (r / 4) + 4 * q + (r % 4);
        const bool ok = row < a.N;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float lik = fam_lik<FAM>(a.L, acc[g][t][r], yv[g][r]);
          sacc[t] += ok ? (double)lik : 0.0;
        }
      }
  }

  // Lanes l and l ^ 32 hold the same chain; then waves in order; then blocks.
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    sacc[t] += __shfl_xor(sacc[t], 32, kWave);
    if (q == 0) lds_red[w][32 * t + rsub] = sacc[t];
  }
  __syncthreads();
  if (threadIdx.x < 32 * NT) {
    double s = 0.0;
    for (int v = 0; v < kFcWaves; ++v) s += lds_red[v][threadIdx.x];
    publish(a.partial + (int64_t)blockIdx.x * kFcChainsMax + threadIdx.x, s);
  }
  if (!arrive_last(a.counter, gridDim.x, &flag)) return;
  finish_chains(a, lds_red);
}

// Split-fp16 variant. Each scaled value v = 2^e x (|v| < 2^14) becomes hi = f16(v) and
// lo = f16(v - hi), which hold v to 2^-22 relative; a product is taken as
// lo_x hi_t + hi_x lo_t + hi_x hi_t on the fp16 matrix cores
// (v_mfma_f32_32x32x16_f16, fp32 accumulation; every fp16 product is exact in fp32),
// dropping lo_x lo_t (below 2^-20 of the product). The row dot products are then good
// to about 1e-6 relative where float32 products give 6e-8, for a fifth of the
// matrix-core time of v_mfma_f32_32x32x2_f32. X is read as float32 and split in
// registers; X is scaled by the caller's 2^x_exp (one exponent for the dataset), Theta per
// chain by 2^e_c from max |theta_c| over its finite entries; z = acc 2^-(x_exp + e_c) is
// exact.
//
// Layout: the columns are shared out over S of a block's eight wavefronts (`per` k-blocks
// of 16 columns each, at most KB), and S wavefronts together take a tile of 32 rows, 8 / S
// tiles at a time. Theta's halves for a wavefront's columns stay in its registers for the
// whole launch: lane l holds Theta[32 t + l % 32][16 j + 8 (l / 32) + 0..7] of k-block j and
// chain tile t. X is loaded as it lies in memory, 256 bytes of four rows per instruction, and
// turned into the A operand's order (x[row + l % 32][16 j + 8 (l / 32) + 0..7] on lane l)
// through the wavefront's own 8 KiB of LDS, chunks swizzled by row against bank conflicts;
// the loads of the next AHEAD steps are in flight while a tile is multiplied, across the
// barrier too. (Loading operand order straight from memory touches every cache line with
// four instructions of 32 lines each and stopped at 4.5 TB/s.) With S > 1 a tile
// passes from wavefront to wavefront: in turn i wavefront w multiplies its columns of tile
// i - w onto the accumulators that wavefront w - 1 left in the same LDS (double buffered, one
// barrier per step), so a row's products are added in column order on one accumulator; the
// S wavefronts then share the likelihoods of the tile that the last one has finished.
// (Partial sums of all S wavefronts on one tile, added at the end, save the S - 1 turns of
// filling but round differently: 2e-9 of a potential of 7000 rows.)
// With Theta's operands in LDS instead (128 KiB, one block per unit, each
// wavefront its own rows in operand order): N = 1e6, D = 512, 64 chains 521 -> 432 us, 20
// chains 507 -> 347 (5.9 TB/s of X); N = 400000, D = 1000, 64 chains 1375 -> 615; N = 300007,
// D = 90, 20 chains 107 -> 36; N = 5000 69 -> 14. At 64 chains the partials' LDS traffic and
// the likelihoods add to the read; at D = 30 (74 us for 20 of rows) the likelihoods bound it.
constexpr int kTile = 32;  // rows per tile

// hi = f16(sc v), lo = f16(sc v - hi): sc is a power of two, so both are one rounding of an
// exact value and one mixed-precision fused multiply-add each.
__device__ __forceinline__ void split8(v4f a, v4f b, float sc, f16x8& hi, f16x8& lo) {
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) hi[i] = (_Float16)__builtin_fmaf(v[i], sc, 0.0f);
#pragma unroll
  for (int i = 0; i < 8; ++i) lo[i] = (_Float16)__builtin_fmaf(v[i], sc, -(float)hi[i]);
}

template <int KB, int S, int NT, int FAM>
__global__ void __launch_bounds__(kFcThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
glm_full_chains_split_kernel(FcArgs a) {
  constexpr int kGroups = kFcWaves / S;       // tiles of a block at a time
  // A tile is loaded and multiplied in steps of up to four k-blocks; AHEAD steps of loads
  // are in flight (as the registers beside Theta's allow).
  constexpr int KL = 4, kSteps = KB / KL;
  constexpr int AHEAD = 2;
  constexpr int kSlots = S > 1 ? 2 : 1;
  __shared__ v4f part[kSlots][kFcWaves][kTile * 16];
  __shared__ double lds_red[kFcWaves][kFcChainsMax];
  __shared__ float lds_sc[kFcChainsMax];
  __shared__ float lds_inv[kFcChainsMax];
  __shared__ int flag;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int rsub = lane & 31;
  const int q = lane >> 5;
  const int grp = w / S, wp = w % S;

  // Per-chain exponent: eight threads per chain find max |theta_c| over finite entries.
  {
    const int c = threadIdx.x >> 3, sub = threadIdx.x & 7;
    float m = 0.0f;
    if (c < a.nchains) {
      const float* th = a.thetas + (int64_t)c * a.ld_theta;
      for (int k0 = sub; k0 < a.D; k0 += 64) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = fabsf(th[min(k0 + 8 * i, a.D - 1)]);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (v[i] <= 3.0e38f) m = fmaxf(m, v[i]);
      }
    }
    m = fmaxf(m, __shfl_xor(m, 1, kWave));
    m = fmaxf(m, __shfl_xor(m, 2, kWave));
    m = fmaxf(m, __shfl_xor(m, 4, kWave));
    if (sub == 0) {
      int E = 0;
      if (m > 0.0f) frexpf(m, &E);  // m < 2^E
      const int e = min(64, max(-64, 14 - E));
      lds_sc[c] = ldexpf(1.0f, e);
      lds_inv[c] = ldexpf(1.0f, -(e + a.x_exp));
    }
  }
  __syncthreads();

  // This wavefront's k-blocks j0 .. j0 + nk - 1 and their Theta operands.
  const int D16 = (a.D + 15) / 16;
  const int per = (D16 + S - 1) / S;  // <= KB
  const int j0 = wp * per;
  const int nk = max(0, min(per, D16 - j0));
  f16x8 bh[KB][NT], bl[KB][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = 32 * t + rsub;
    const bool live = c < a.nchains;
    const float* src = a.thetas + (int64_t)(live ? c : 0) * a.ld_theta;
    const float sc = lds_sc[c];
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      const int k0 = 16 * (j0 + u) + 8 * q;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool ok = live && u < nk && k0 + i < a.D;
        const float x = src[ok ? k0 + i : 0];
        const float v = ok ? x * sc : 0.0f;
        const _Float16 h = (_Float16)v;
        bh[u][t][i] = h;
        bl[u][t][i] = (_Float16)(v - (float)h);
      }
    }
  }
  const float xs = ldexpf(1.0f, a.x_exp);
  float inv[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) inv[t] = lds_inv[32 * t + rsub];
  // Tiles of the block, dealt to its groups in turn; every group makes `turns` passes (the
  // barriers are the block's), the last ones on tiles past t1 whose rows count for nothing.
  const int64_t t0 = (int64_t)blockIdx.x * a.tiles / gridDim.x;
  const int64_t t1 = (int64_t)(blockIdx.x + 1) * a.tiles / gridDim.x;
  const int turns = (int)((t1 - t0 + kGroups - 1) / kGroups);
  double sacc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) sacc[t] = 0.0;

  // Instruction i of a step loads rows 4 i + l / 16 of the tile, lane l the 16-byte chunk
  // c = (l % 16) ^ (row % 16) of the wavefront's 16 (its LDS place is then l % 16), through a
  // buffer resource that begins at the tile and ends with the data: rows past N read as
  // zero, and chunks that are not the wavefront's or not the row's lie past its end (kOut).
  constexpr uint32_t kOut = 0x80000000u;
  v4f x[AHEAD][8];
  const int lrow = lane >> 4;
  uint32_t voff[kSteps][4];
#pragma unroll
  for (int h = 0; h < kSteps; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = (lane & 15) ^ (4 * i + lrow);
      const int c4 = 4 * (j0 + KL * h) + c;
      voff[h][i] = c < 4 * (nk - KL * h) && c4 < a.D4
                       ? (uint32_t)(lrow * a.ldx + 4 * c4) * 4u : kOut;
    }
  const uint32_t row4 = (uint32_t)(16 * a.ldx);  // bytes of four rows
  auto resource = [&](const float* base, int64_t left) __attribute__((always_inline)) {
    const int64_t bytes = max((int64_t)0, min(4 * left, (int64_t)0x7FFFFFFF));
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
  };
  auto load = [&](int step, auto hh, v4f (&buf)[8]) __attribute__((always_inline)) {
    constexpr int H = decltype(hh)::value;
    const int turn = step / kSteps - wp;  // (outside the block's turns: no rows)
    const int64_t row0 = turn < 0 || turn >= turns
                             ? a.N : (t0 + (int64_t)turn * kGroups + grp) * kTile;
    const auto rs = resource(a.X + min(row0, a.N) * a.ldx, (a.N - row0) * a.ldx);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      buf[i] = __builtin_bit_cast(
          v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[H][i & 3] + i * row4, 0, 0));
  };
  // likelihood of accumulator quad qd (rows 8 (qd % 4) + 4 q + 0..3, chain tile qd / 4)
  auto count = [&](int64_t tile, int qd, int t, const float (&z)[4], v4f yv)
                   __attribute__((always_inline)) {
    const bool whole = tile < t1 && tile * kTile + kTile <= a.N;  // uniform
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double lik = (double)fam_lik<FAM>(a.L, z[i] * inv[t], yv[i]);
      if (whole) sacc[t] += lik;
      else sacc[t] += tile < t1 && tile * kTile + 8 * (qd % 4) + 4 * q + i < a.N ? lik : 0.0;
    }
  };
  constexpr int kQuads = S >= 4 * NT ? 1 : 4 * NT / S;  // per wavefront
  v16f acc[NT];
  v4f yv[kQuads];
  const bool ragged = (a.D & 3) != 0 && nk > 0 && j0 + nk == D16;  // uniform
  // step `step` (its place H in the tile static); its loads are in cur, which then takes
  // those of step + AHEAD
  auto step_of = [&](int step, auto hh, v4f (&cur)[8]) __attribute__((always_inline)) {
    constexpr int H = decltype(hh)::value;
    // the tile that the last of the S wavefronts finishes in this turn
    const int turn = step / kSteps - (S - 1);
    const int64_t tile = t0 + (int64_t)turn * kGroups + grp;
    v4f* mine = part[step & (kSlots - 1)][w];
    if (ragged) {
      // columns past D in the row's last chunk: a scaled padding value could overflow fp16,
      // and inf times Theta's zero is NaN
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int c = (lane & 15) ^ ((4 * i + lrow) & 15);
        if (4 * (j0 + KL * H) + c == a.D4 - 1) {
          if ((a.D & 3) == 1) cur[i].y = 0.0f;
          if ((a.D & 3) <= 2) cur[i].z = 0.0f;
          cur[i].w = 0.0f;
        }
      }
    }
    wave_sync();  // the step before has read the slot
#pragma unroll
    for (int i = 0; i < 8; ++i) mine[i * kWave + lane] = cur[i];
    wave_sync();
    load(step + AHEAD, std::integral_constant<int, (H + AHEAD) % kSteps>{}, cur);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
    if (H == 0) {
      const int64_t row0 = turn < 0 ? a.N : tile * kTile;
      const auto ys = resource(a.y + min(row0, a.N), a.N - row0);
#pragma unroll
      for (int i = 0; i < kQuads; ++i)
        yv[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                            ys, 32 * ((wp + i * S) % 4) + 16 * q, 0, 0));
      if (S == 1 || wp == 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = v16f{};
      } else {  // go on from the wavefront before, which had this tile in the turn before
        const v4f* prev = part[(step - 1) & (kSlots - 1)][w - 1];
#pragma unroll
        for (int qd = 0; qd < 4 * NT; ++qd) {
          const v4f v = prev[qd * kWave + lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[qd / 4][4 * (qd % 4) + i] = v[i];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < KL; ++u) {
      if (KL * H + u >= nk) break;
      f16x8 ah, al;
      const int c = 4 * u + 2 * q, r = rsub & 15;
      split8(mine[rsub * 16 + (c ^ r)], mine[rsub * 16 + ((c + 1) ^ r)], xs, ah, al);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[KL * H + u][t], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[KL * H + u][t], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[KL * H + u][t], acc[t], 0, 0, 0);
    }
    if constexpr (H < kSteps - 1) {
      if (S > 1) lds_sync();  // the slot's partials of the tile before have been read
      return;
    }
    if constexpr (S == 1) {
#pragma unroll
      for (int qd = 0; qd < 4 * NT; ++qd) {
        const float z[4] = {acc[qd / 4][4 * (qd % 4)], acc[qd / 4][4 * (qd % 4) + 1],
                            acc[qd / 4][4 * (qd % 4) + 2], acc[qd / 4][4 * (qd % 4) + 3]};
        count(tile, qd, qd / 4, z, yv[qd]);
      }
    } else {
      auto& buf = part[step & 1];
#pragma unroll
      for (int qd = 0; qd < 4 * NT; ++qd)
        mine[qd * kWave + lane] = v4f{acc[qd / 4][4 * (qd % 4)], acc[qd / 4][4 * (qd % 4) + 1],
                                      acc[qd / 4][4 * (qd % 4) + 2], acc[qd / 4][4 * (qd % 4) + 3]};
      lds_sync();  // what this slot is used for next lies behind the next step's barrier
      if (turn < 0) return;
#pragma unroll
      for (int i = 0; i < kQuads; ++i) {
        const int qd = wp + i * S;
        if (qd >= 4 * NT) break;
        const v4f s = buf[grp * S + S - 1][qd * kWave + lane];
        const float z[4] = {s.x, s.y, s.z, s.w};
        // (the chain tile of quad wp + i S; uniform, a register index needs it static)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (qd / 4 == t) count(tile, qd, t, z, yv[i]);
      }
    }
  };
  static_assert(AHEAD == 2, "the two steps below");
  load(0, std::integral_constant<int, 0>{}, x[0]);
  load(1, std::integral_constant<int, 1 % kSteps>{}, x[1]);
  // AHEAD kSteps steps per round, so that buffers and places in the tile are static
  const int steps = (turns + S - 1) * kSteps;
  auto round = [&](int base, auto self, auto bb) __attribute__((always_inline)) {
    constexpr int B = decltype(bb)::value;
    if (base + B < steps)
      step_of(base + B, std::integral_constant<int, B % kSteps>{}, x[B % AHEAD]);
    if constexpr (B + 1 < AHEAD * kSteps) self(base, self, std::integral_constant<int, B + 1>{});
  };
  for (int base = 0; base < steps; base += AHEAD * kSteps)
    round(base, round, std::integral_constant<int, 0>{});

  // Lanes l and l ^ 32 hold the same chain; then waves in order; then blocks.
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    sacc[t] += __shfl_xor(sacc[t], 32, kWave);
    if (q == 0) lds_red[w][32 * t + rsub] = sacc[t];
  }
  __syncthreads();
  if (threadIdx.x < 32 * NT) {
    double sum = 0.0;
    for (int v = 0; v < kFcWaves; ++v) sum += lds_red[v][threadIdx.x];
    publish(a.partial + (int64_t)blockIdx.x * kFcChainsMax + threadIdx.x, sum);
  }
  if (!arrive_last(a.counter, gridDim.x, &flag)) return;
  finish_chains(a, lds_red);
}

}  // namespace
}  // namespace sgmc

using namespace sgmc;

namespace {

// The wavefronts that share a row's columns: as few as hold them in KB = 4 k-blocks of
// registers each; all eight with 8 k-blocks each (and one chain tile) beyond 512 columns.
template <int FAM>
void launch_split(dim3 grid, hipStream_t s, const FcArgs& a, int D16, bool two) {
  const dim3 block(kFcThreads);
#define SGMC_SPLIT(KB, S, NT) \
  hipLaunchKernelGGL((glm_full_chains_split_kernel<KB, S, NT, FAM>), grid, block, 0, s, a)
  if (D16 <= 4) {
    if (two) SGMC_SPLIT(4, 1, 2);
    else SGMC_SPLIT(4, 1, 1);
  } else if (D16 <= 8) {
    if (two) SGMC_SPLIT(4, 2, 2);
    else SGMC_SPLIT(4, 2, 1);
  } else if (D16 <= 16) {
    if (two) SGMC_SPLIT(4, 4, 2);
    else SGMC_SPLIT(4, 4, 1);
  } else if (D16 <= 32) {
    if (two) SGMC_SPLIT(4, 8, 2);
    else SGMC_SPLIT(4, 8, 1);
  } else {
    SGMC_SPLIT(8, 8, 1);
  }
#undef SGMC_SPLIT
}

int launch_full_chains(const char* name, bool split, int x_exp, int family, const float* X,
                       int64_t ldx, const float* y, int64_t N, int D, const float* thetas,
                       int64_t ld_theta, int nchains, float sigma, int has_prior,
                       float prior_scale, double temperature, double* out_U, double* workspace,
                       int64_t workspace_doubles, int nblocks, void* stream) {
  SGMC_REQUIRE(X && y && thetas && out_U && workspace, SGMC_E_ARG, "%s: null pointer", name);
  SGMC_REQUIRE(family == SGMC_LIK_LINEAR_GAUSSIAN || family == SGMC_LIK_LOGISTIC, SGMC_E_ARG,
               "%s: unknown family %d", name, family);
  SGMC_REQUIRE(D >= 1 && D <= 1024, SGMC_E_ARG, "%s: D=%d outside [1, 1024]", name, D);
  SGMC_REQUIRE(ldx % 4 == 0 && ldx >= 4 * ((D + 3) / 4), SGMC_E_ARG,
               "%s: ldx must be a multiple of 4 and >= D rounded up", name);
  SGMC_REQUIRE(((uintptr_t)X & 15) == 0, SGMC_E_ARG, "%s: X not 16-byte aligned", name);
  SGMC_REQUIRE(ld_theta >= D, SGMC_E_ARG, "%s: ld_theta < D", name);
  SGMC_REQUIRE(N >= 1 && nchains >= 1 && nblocks >= 1, SGMC_E_ARG, "%s: bad size", name);
  SGMC_REQUIRE(workspace_doubles >= sgmc_glm_full_chains_workspace_doubles(nblocks), SGMC_E_ARG,
               "%s: workspace too small", name);
  SGMC_REQUIRE(temperature != 0.0, SGMC_E_ARG, "%s: temperature is zero", name);
  SGMC_REQUIRE(x_exp >= -64 && x_exp <= 64, SGMC_E_ARG, "%s: x_exp=%d outside [-64, 64]", name,
               x_exp);
  // The split kernel reaches the rows of a tile by 31-bit byte offsets from its first row:
  // 31 rows on and a row's columns further. Longer strides (over about 17.3 M floats: a column
  // slice of a very wide matrix) take the float32 kernel, which addresses every row in 64 bits.
  const bool far = (kTile - 1) * 4 * ldx + 16 * (int64_t)((D + 3) / 4) > 0x7FFFFFFF;
  split = split && !far;
  FcArgs a;
  a.X = X;
  a.y = y;
  a.ldx = ldx;
  a.ld_theta = ld_theta;
  a.N = N;
  a.tiles = split ? (N + kTile - 1) / kTile : (N + 63) / 64;
  a.D = D;
  a.D4 = (D + 3) / 4;
  const int D8 = (D + 7) / 8;
  a.D8r = (D8 + kFcAhead - 1) / kFcAhead * kFcAhead;
  const int D16 = (D + 15) / 16;
  a.x_exp = x_exp;
  a.L = make_lik(family, sigma);
  a.pr = make_prior(has_prior, prior_scale);
  a.temperature = temperature;
  a.partial = workspace;
  a.counter = reinterpret_cast<unsigned*>(workspace + (int64_t)nblocks * kFcChainsMax);
  // Two chain tiles per pass when their operands fit the LDS (split: the registers), else
  // one.
  const int nt = split ? (D16 <= 32 ? 2 : 1) : ((a.D8r * 2 * kWave <= kFcLdsF4) ? 2 : 1);
  hipStream_t s = as_stream(stream);
  const dim3 grid(nblocks), block(kFcThreads);
  for (int c0 = 0; c0 < nchains; c0 += 32 * nt) {
    a.thetas = thetas + (int64_t)c0 * ld_theta;
    a.out_U = out_U + c0;
    a.nchains = nchains - c0 < 32 * nt ? nchains - c0 : 32 * nt;
    const bool two = a.nchains > 32;
    const bool lg = family == SGMC_LIK_LOGISTIC;
    if (split) {
      if (lg) launch_split<SGMC_LIK_LOGISTIC>(grid, s, a, D16, two);
      else launch_split<SGMC_LIK_LINEAR_GAUSSIAN>(grid, s, a, D16, two);
    } else {
      if (lg) {
        if (two) hipLaunchKernelGGL((glm_full_chains_kernel<2, SGMC_LIK_LOGISTIC>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((glm_full_chains_kernel<1, SGMC_LIK_LOGISTIC>), grid, block, 0, s, a);
      } else {
        if (two) hipLaunchKernelGGL((glm_full_chains_kernel<2, SGMC_LIK_LINEAR_GAUSSIAN>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((glm_full_chains_kernel<1, SGMC_LIK_LINEAR_GAUSSIAN>), grid, block, 0, s, a);
      }
    }
    const int rc = check_launch(name);
    if (rc != SGMC_OK) return rc;
  }
  return SGMC_OK;
}

}  // namespace

extern "C" {

int64_t sgmc_glm_full_chains_workspace_doubles(int nblocks) {
  return (int64_t)nblocks * kFcChainsMax + 2;
}

int sgmc_glm_full_potential_chains(int family, const float* X, int64_t ldx, const float* y,
                                   int64_t N, int D, const float* thetas, int64_t ld_theta,
                                   int nchains, float sigma, int has_prior, float prior_scale,
                                   double temperature, double* out_U, double* workspace,
                                   int64_t workspace_doubles, int nblocks, void* stream) {
  return launch_full_chains("sgmc_glm_full_potential_chains", false, 0, family, X, ldx, y, N, D,
                            thetas, ld_theta, nchains, sigma, has_prior, prior_scale,
                            temperature, out_U, workspace, workspace_doubles, nblocks, stream);
}

int sgmc_glm_full_potential_chains_split(int family, const float* X, int64_t ldx,
                                         const float* y, int64_t N, int D, const float* thetas,
                                         int64_t ld_theta, int nchains, float sigma,
                                         int has_prior, float prior_scale, double temperature,
                                         int x_exp, double* out_U, double* workspace,
                                         int64_t workspace_doubles, int nblocks, void* stream) {
  return launch_full_chains("sgmc_glm_full_potential_chains_split", true, x_exp, family, X, ldx,
                            y, N, D, thetas, ld_theta, nchains, sigma, has_prior, prior_scale,
                            temperature, out_U, workspace, workspace_doubles, nblocks, stream);
}

}  // extern "C"
