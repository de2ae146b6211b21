// Bayesian MLP classifier likelihood on MFMA (bf16 operands, fp32 accumulation), with
// a hand-written backward pass and the SGLD / rms_prop update fused into the weight-
// gradient GEMM epilogue. Model (the likelihood a user writes in the reference as
// likelihood(sample, obs), potential.py:128-137):
//   h1 = relu(x W1 + b1), h2 = relu(h1 W2 + b2), logits = h2 W3 + b3,
//   lik = log_softmax(logits)[label]
// Parameters are one float32 vector per chain in tree_flatten order of
// {"W1","W2","W3","b1","b2","b3"} (sorted keys): W1 [D_in][H1], W2 [H1][H2],
// W3 [H2][10], b1, b2, b3. A bf16 shadow of the parameters (same layout) feeds the
// GEMMs and is rewritten by every update.
//
// One step for C chains (grid z = chain), potential U = (-N mean(lik) - log p)/T with
// a Gaussian prior, gradient by back-propagation:
//   gather   Xb = bf16(X[idx]) (index draw in-kernel, data/numpy_loader.py:132-134)
//   G1       H1 = relu(Xb W1 + b1)
//   G2       H2 = relu(H1 W2 + b2)
//   head     logits, softmax, lik, dL = c (onehot - p), dA2 = (dL W3^T) * (H2 > 0)
//   G3       dA1 = (dA2 W2^T) * (H1 > 0)
//   G4       gW2 = H1^T dA2  -> update W2 in the epilogue
//   G5       gW1 = Xb^T dA1  -> update W1 in the epilogue
//   small    W3, b1, b2, b3 gradients and updates; U; key and data-key advance
// c = -N / (n T) carries the potential's scaling into the backward pass.
//
// Precisions: bf16 GEMM operands (v_mfma_f32_32x32x16_bf16), OCP e4m3 with per-tensor
// scales (v_mfma_f32_32x32x16_fp8_fp8), or float32 (v_mfma_f32_32x32x2_f32: activations
// stored in float32, weights read from theta itself, no shadow); fp32 accumulation in
// all three.
//
// The GEMMs: mlp_fwd.hip (G1-G3) and mlp_param.hip (G4, G5 with the update, beside the small
// leaves' column sums of mlp_colsum.h).
#include <math.h>

#include <type_traits>

#include "mlp_update.h"

namespace sgmc {
namespace mlp {

#ifndef SGMC_GATHER_BATCH
#define SGMC_GATHER_BATCH 12
#endif
constexpr int kGatherBatch = SGMC_GATHER_BATCH;  // float4 row loads in flight per lane
// Gradient-only variant: grad = (gsum + prior) / T, no update.
__device__ __forceinline__ void grad_param(const Step& s, const float* th, float* gout,
                                           int64_t i, float gsum, float& lp) {
  const float w = th[i];
  float g = gsum;
  if (s.has_prior) {
    g = g + w * s.prior_inv_var;
    lp += (s.prior_log_norm + (w * w) * s.prior_inv_var) / -2.0f;
  }
  gout[i] = g / s.temperature;
}


// ------------------------------------------------------------------ gather ----
// Xb[c][j] = bf16(X[idx_j]), lab[c][j] = labels[idx_j]; one wavefront per row,
// ROWS rows per block.
// What bounds it: the rows' HBM reads (16 x 512 rows of 3072: 100 MB, 16 us at the 6.5 TB/s
// of a random gather, 32 us measured behind an update's stores). The block's first
// wavefront draws all its indices (five dependent Threefry blocks each, 500 instructions
// that every wavefront ran for its own row), the e4m3 maximum costs a block one atomic at
// most (with one per wavefront 512 of them queued on each chain's word: 67 us), and a
// minibatch's rows are read with the non-temporal hint, which leaves the last-level cache
// to the weights (16 x 256 rows: 24 -> 19 us, and the Xb W1 that follows 36 -> 30 us).
// FULL: the rows of a full-data pass, the same for all chains; a wavefront reads its row
// once for kGatherChains of them (16 x 512 rows: 10.9 us, with 1 chain 11.9, with 4 11.3).
constexpr int kGatherChains = 2;
template <bool FULL, int ROWS>
__global__ void __launch_bounds__(ROWS* kWave) gather_kernel(Step s) {
  __shared__ int64_t rows[ROWS];
  __shared__ float red[ROWS];
  __shared__ double red_d[ROWS];
  const int c0 = blockIdx.y * (FULL ? kGatherChains : 1);
  const int c1 = FULL ? min(c0 + kGatherChains, s.C) : c0 + 1;
  if (s.update && !FULL && blockIdx.x == 0 && threadIdx.x < NLEAF)
    store_key(s.lkey + 2 * (c0 * NLEAF + threadIdx.x), derive_leaf_key(s, c0, threadIdx.x));
  const int w = threadIdx.x / kWave;
  const int j = blockIdx.x * ROWS + w;  // s.n is a multiple of ROWS
  const int lane = threadIdx.x & (kWave - 1);
  int64_t r;
  bool valid = true;
  if (FULL) {  // rows row0 + j of the full-data pass; rows past N are zero
    r = s.row0 + j;
    valid = r < s.N;
    if (!valid) r = 0;
  } else {
    if (threadIdx.x < ROWS) {
      Key next, sub, k1, k2;
      split2(load_key(s.dkey + 2 * c0), next, sub);
      split2(sub, k1, k2);
      const uint32_t span = (uint32_t)s.N;
      r = (int64_t)draw_index(k1, k2, (uint32_t)s.n,
                              (uint32_t)(blockIdx.x * ROWS + threadIdx.x), span, s.rmult,
                              s.rmagic);
      if (r < 0 || r >= s.N) r = 0;
      rows[threadIdx.x] = r;
    }
    lds_sync();
    r = rows[w];
  }
  const float* __restrict__ src = s.X + r * s.ldx;
  // kGatherBatch float4 loads per lane go out before their conversions and stores, so a
  // row costs D_in / (256 kGatherBatch) memory round trips instead of D_in / 256. The
  // loads are unconditional: offsets past the row are clamped to its last float4 (and
  // not stored), a row past N reads row 0 and is zeroed.
  constexpr int kStep = kWave * 4;
  const f32x4 zero4{0.f, 0.f, 0.f, 0.f};
  auto rowcopy = [&](auto&& put) __attribute__((always_inline)) {
    for (int f0 = lane * 4; f0 < s.D_in; f0 += kGatherBatch * kStep) {
      f32x4 xs[kGatherBatch];
#pragma unroll
      for (int u = 0; u < kGatherBatch; ++u) {
        const f32x4* p = reinterpret_cast<const f32x4*>(src + min(f0 + u * kStep, s.D_in - 4));
        if constexpr (FULL) xs[u] = *p;
        else xs[u] = __builtin_nontemporal_load(p);
      }
#pragma unroll
      for (int u = 0; u < kGatherBatch; ++u) xs[u] = valid ? xs[u] : zero4;
      for (int c = c0; c < c1; ++c) {
        const int64_t row = ((int64_t)c * s.n + j) * s.D_in;
        const float qs = s.fp8 ? s.q[(int64_t)c * kQWords + Q_X] : 1.0f;
#pragma unroll
        for (int u = 0; u < kGatherBatch; ++u)
          if (f0 + u * kStep < s.D_in) put(row + f0 + u * kStep, xs[u], qs);
      }
    }
  };
  if (s.fp8) {
    uint8_t* __restrict__ dst = reinterpret_cast<uint8_t*>(s.Xb);
    float amax = 0.f;
    rowcopy([&](int64_t i, f32x4 x, float qs) {
      amax = fmaxf(amax, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
      *reinterpret_cast<uint32_t*>(dst + i) = pack_q(x * qs);
    });
    if constexpr (FULL)
      for (int c = c0; c < c1; ++c) q_note_amax(s, c, Q_X, amax);
    else
      q_note_amax_block(s, c0, Q_X, amax, red);
  } else if (s.fp32) {
    float* __restrict__ dst = reinterpret_cast<float*>(s.Xb);
    rowcopy([&](int64_t i, f32x4 x, float) { *reinterpret_cast<f32x4*>(dst + i) = x; });
  } else {
    uint16_t* __restrict__ dst = reinterpret_cast<uint16_t*>(s.Xb);
    rowcopy([&](int64_t i, f32x4 x, float) {
      *reinterpret_cast<u32x2_4*>(dst + i) = pack_bf(x);
    });
  }
  if constexpr (FULL) {
    // the chunk before this one: its likelihoods, which the head behind this launch
    // overwrites, go to the pass's float64 sum (fixed order); the first chunk clears it
    if (blockIdx.x == 0) {
      for (int c = c0; c < c1; ++c) {
        double t = 0.0;
        if (s.row0 > 0)
          for (int i = threadIdx.x; i < s.n; i += ROWS * kWave)
            t += (double)s.lik[(int64_t)c * s.n + i];
        t = block_sum_d<ROWS * kWave>(t, red_d);
        if (threadIdx.x == 0) s.facc[c] = s.row0 > 0 ? s.facc[c] + t : 0.0;
      }
    }
  }
  if (lane == 0)
    for (int c = c0; c < c1; ++c) s.lab[(int64_t)c * s.n + j] = valid ? s.labels[r] : -1;
}

// ------------------------------------------------------------------ head ------
// logits = h2 W3 + b3; p = softmax; lik = logits[label] - lse; dL = c (onehot - p);
// dA2 = (dL W3^T) * (h2 > 0). A wavefront takes R rows of one chain. W3S: W3 is staged in
// LDS (row stride kW3Stride, so lanes reading consecutive rows of W3 hit distinct banks)
// and each W3 row read serves all of the wavefront's rows; otherwise W3 comes from global
// memory. For every row the sums run in the same order either way: lane-partial sums
// over the columns a = lane + 64 u in ascending u, then wave sums.
// What bounds it: latency, then the vector ALU (8192 rows of H2 = 1024 read 17 MB, 3.3 us,
// and take 4.3 us of multiplies and adds). So a batch of h2 is always in flight (the first
// behind the staging of W3), the 10 R sums of a wavefront share their lane swaps (100
// instructions for 40 sums where 40 separate ones take 320), and the softmax of row r runs
// on lane r instead of R times on all: 36 -> 13 us per launch (4096 rows of H2 = 512: 16 ->
// 10 us).
constexpr int kW3Stride = NCLS + 1;

// h2 element as loaded (bf16 or float32) and its value; the ReLU mask of the raw element.
template <bool F32>
__device__ __forceinline__ uint32_t h2_raw(const void* h2, int64_t i) {
  if (F32) return reinterpret_cast<const uint32_t*>(h2)[i];
  return reinterpret_cast<const uint16_t*>(h2)[i];
}
template <bool F32>
__device__ __forceinline__ float h2_val(uint32_t raw) {
  return __uint_as_float(F32 ? raw : raw << 16);
}
template <bool F32>
__device__ __forceinline__ bool h2_on(uint32_t raw) {
  return raw != 0 && !(raw & (F32 ? 0x80000000u : 0x8000u));
}

template <int PREC, bool W3S, int R, int NW>
__global__ void __launch_bounds__(kWave* NW) head_kernel(Step s) {
  constexpr bool F32 = PREC == P_F32;
  constexpr int NB = 4;             // columns per lane and batch
  constexpr int kZ = R * NCLS;      // logits of a wavefront
  constexpr int kZ4 = (kZ + 3) / 4 * 4;
  extern __shared__ float w3s[];    // W3S: [H2][kW3Stride]
  __shared__ __attribute__((aligned(16))) float zs[NW][kZ4];
  __shared__ float red[NW];
  const int c = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const float* th = s.theta + (int64_t)c * s.P;
  const float* W3 = th + s.off[2];
  const float* b3 = th + s.off[5];
  const int U = s.H2 / kWave;       // columns per lane (a multiple of 2)
  const int j0 = (blockIdx.x * NW + wv) * R;  // s.n is a multiple of NW R
  const int64_t row0 = (int64_t)c * s.n + j0;
  uint32_t nx[R][NB];
  auto fetch = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < NB; ++u)
        nx[r][u] = h2_raw<F32>(s.h2, (row0 + r) * s.H2 + lane + min(u0 + u, U - 1) * kWave);
  };
  fetch(0);
  if (W3S) {
    // 16 loads per thread go out before their LDS stores (indices past W3 are clamped
    // to its last element and not stored)
    constexpr int kNT = kWave * NW;
    const int total = s.H2 * NCLS;
    for (int i0 = threadIdx.x; i0 < total; i0 += 16 * kNT) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = W3[min(i0 + u * kNT, total - 1)];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int i = i0 + u * kNT;
        if (i < total) w3s[(i / NCLS) * kW3Stride + i % NCLS] = v[u];
      }
    }
    lds_sync();
  }
  auto w3at = [&](int a, int k) __attribute__((always_inline)) -> float {
    return W3S ? w3s[a * kW3Stride + k] : W3[(int64_t)a * NCLS + k];
  };
  float z[kZ4];
#pragma unroll
  for (int i = 0; i < kZ4; ++i) z[i] = 0.f;
  for (int u0 = 0; u0 < U; u0 += NB) {
    uint32_t h[R][NB];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < NB; ++u) h[r][u] = nx[r][u];
    fetch(u0 + NB < U ? u0 + NB : 0);  // at the end: the masks' first batch
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (u == 2 && u0 + 2 >= U) break;
      float w[NCLS];
#pragma unroll
      for (int k = 0; k < NCLS; ++k) w[k] = w3at(lane + (u0 + u) * kWave, k);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < NCLS; ++k) z[r * NCLS + k] += h2_val<F32>(h[r][u]) * w[k];
    }
  }
  // The wavefront sums of the kZ logits, the additions of wave_sum: the xor-32 and xor-16
  // steps of two values share a lane swap, which leaves in row of 16 g, register j the
  // value 4 j + 2 (g % 2) + g / 2.
  float q[kZ4 / 4];
  {
    float p[kZ4 / 2];
#pragma unroll
    for (int i = 0; i < kZ4 / 2; ++i) p[i] = pair_add32(z[2 * i], z[2 * i + 1]);
#pragma unroll
    for (int j = 0; j < kZ4 / 4; ++j) q[j] = pair_add16(p[2 * j], p[2 * j + 1]);
  }
#pragma unroll
  for (int j = 0; j < kZ4 / 4; ++j)
    q[j] = ror_add<1>(ror_add<2>(ror_add<4>(ror_add<8>(q[j]))));
  if ((lane & 15) == 0) {
    const int g = lane >> 4;
#pragma unroll
    for (int j = 0; j < kZ4 / 4; ++j) zs[wv][4 * j + 2 * (g & 1) + (g >> 1)] = q[j];
  }
  wave_sync();
  // lane r: softmax of row r (a wavefront's LDS accesses complete in order)
  const float cscale = ((float)(-s.N) / (float)s.n) / s.temperature;
  if (lane < R) {
    float zr[NCLS];
#pragma unroll
    for (int k = 0; k < NCLS; ++k) zr[k] = zs[wv][lane * NCLS + k] + b3[k];
    float mx = zr[0];
#pragma unroll
    for (int k = 1; k < NCLS; ++k) mx = fmaxf(mx, zr[k]);
    float se = 0.f;
#pragma unroll
    for (int k = 0; k < NCLS; ++k) se += expf(zr[k] - mx);
    const float lse = mx + logf(se);
    const int lab = s.lab[row0 + lane];
    const int lb = lab < 0 ? 0 : (lab >= NCLS ? NCLS - 1 : lab);
    float zl = zr[0];
#pragma unroll
    for (int k = 1; k < NCLS; ++k)
      if (k == lb) zl = zr[k];
    // the full pass wants the likelihood only; its padding rows (label -1) contribute 0
    s.lik[row0 + lane] = s.full && lab < 0 ? 0.0f : zl - lse;
    if (!s.full) {
#pragma unroll
      for (int k = 0; k < NCLS; ++k) {
        const float d = cscale * ((k == lb ? 1.0f : 0.0f) - expf(zr[k] - lse));
        s.dL[(row0 + lane) * NCLS + k] = d;
        zs[wv][lane * NCLS + k] = d;
      }
    }
  }
  if (s.full) return;
  wave_sync();
  float dl[kZ];
#pragma unroll
  for (int i = 0; i < kZ; ++i) dl[i] = zs[wv][i];
  const float qs = PREC == P_FP8 ? s.q[(int64_t)c * kQWords + Q_DA2] : 1.0f;
  float amax = 0.f;
  for (int u0 = 0; u0 < U; u0 += NB) {
    uint32_t h[R][NB];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < NB; ++u) h[r][u] = nx[r][u];
    if (u0 + NB < U) fetch(u0 + NB);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (u == 2 && u0 + 2 >= U) break;
      const int a = lane + (u0 + u) * kWave;
      float w[NCLS];
#pragma unroll
      for (int k = 0; k < NCLS; ++k) w[k] = w3at(a, k);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float d = 0.f;
#pragma unroll
        for (int k = 0; k < NCLS; ++k) d += dl[r * NCLS + k] * w[k];
        const float v = h2_on<F32>(h[r][u]) ? d : 0.0f;
        amax = fmaxf(amax, fabsf(v));
        put_act(s.da2, (row0 + r) * s.H2 + a, v, PREC == P_FP8, qs, F32);
      }
    }
  }
  if (PREC == P_FP8) q_note_amax_block(s, c, Q_DA2, amax, red);
}

// ----------------------------------------------------------- small params -----
// W3, b1, b2, b3: gradient by a loop over the n rows, update, prior partial; the last
// block of a chain forms U and advances the chain's keys (and the iteration counter
// once every chain is done).
__global__ void __launch_bounds__(GT) small_kernel(Step s, int part0) {
  __shared__ float red[GT / kWave];
  __shared__ double red_d[GT / kWave];
  __shared__ int flag;
  const int c = blockIdx.y;
  const int64_t nW3 = (int64_t)s.H2 * NCLS;
  const int64_t total = nW3 + s.H1 + s.H2 + NCLS;
  const int64_t p = (int64_t)blockIdx.x * GT + threadIdx.x;
  const int it = cur_iter(s);
  const Coef cf = coef_of(s);
  float lp = 0.f, ke = 0.f;
  if (p < total) {
    int leaf;
    int64_t i;
    if (p < nW3) {
      leaf = 2;
      i = p;
    } else if (p < nW3 + s.H1) {
      leaf = 3;
      i = p - nW3;
    } else if (p < nW3 + s.H1 + s.H2) {
      leaf = 4;
      i = p - nW3 - s.H1;
    } else {
      leaf = 5;
      i = p - nW3 - s.H1 - s.H2;
    }
    const int64_t base = (int64_t)c * s.P + s.off[leaf];
    // the parameter's state and its key are in flight with the first strips' sums
    const Upd up = make_upd(s, c, leaf, base, cf);
    float wmax = 0.f, w = 0.f, aux = 0.f;
    Key lk{};
    if (s.update) {
      lk = leaf_key(s, c, leaf);
      upd_load(up, (uint32_t)i, w, aux);
    }
    const int strips = s.n / kStrip;
    const float* cp = s.col_part + (int64_t)c * strips * total + p;
    float gsum = 0.f;
    for (int t = 0; t < strips; t += 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = t + u < strips ? cp[(int64_t)(t + u) * total] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) gsum += x[u];
    }
    if (s.update) {
      const float xi = bits_to_normal_fast(bits_word(lk, (uint32_t)s.size[leaf], (uint32_t)i));
      upd_step(up, w, aux, gsum, xi, lp, ke);
      upd_store(up, (uint32_t)i, w, aux, wmax);
    } else {
      grad_param(s, s.theta + base, s.grad + base, i, gsum, lp);
    }
  }
  const bool obabo = s.update && s.mode != MLP_SGLD;
  const int64_t slot = (int64_t)c * s.nparts + part0 + blockIdx.x;
  const float tot = block_sum<GT>(lp, red);
  if (threadIdx.x == 0) publish(s.prior_part + slot, tot);
  if (obabo) {
    const float kt = block_sum<GT>(ke, red);
    if (threadIdx.x == 0) publish(s.ke_part + slot, kt);
  }
  if (!arrive_last(s.counters + c, gridDim.x, &flag)) return;
  // One memory round trip for all the tail reads: the records and likelihoods go out
  // together, and the next keys are derived behind them.
  Key k_next{}, d_next{};
  double kin = 0.0;
  float lsum = 0.f, prior = 0.f;
  for (int q0 = threadIdx.x; q0 < max(s.nparts, s.n); q0 += 4 * GT) {
    float xk[4], xl[4], xp[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = q0 + u * GT;
      xp[u] = q < s.nparts ? consume(s.prior_part + (int64_t)c * s.nparts + q) : 0.f;
      xk[u] = obabo && q < s.nparts ? consume(s.ke_part + (int64_t)c * s.nparts + q) : 0.f;
      xl[u] = q < s.n ? s.lik[(int64_t)c * s.n + q] : 0.f;
    }
    if (q0 == 0 && s.update) {
      Key a, b;
      const Key k0 = load_key(s.key + 2 * c), d0 = load_key(s.dkey + 2 * c);
      split2(d0, d_next, a);
      if (obabo) split3(k0, k_next, a, b);
      else split2(k0, k_next, a);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      prior += xp[u];
      kin += (double)xk[u];
      lsum += xl[u];
    }
  }
  if (obabo) kin = block_sum_d<GT>(kin, red_d);
  lsum = block_sum<GT>(lsum, red);
  prior = block_sum<GT>(prior, red);
  if (threadIdx.x == 0) {
    const float mean = lsum / (float)s.n;
    const float Uc = ((float)(-s.N) * mean - prior) / s.temperature;
    if (obabo) {
      // ObaboState bookkeeping (integrator.py:203-273): the step's potential is the mean
      // of its two evaluations; the key advances once per step, the data key per draw.
      store_key(s.dkey + 2 * c, d_next);
      if (s.mode == MLP_OBABO_BA) {
        s.U_half[c] = Uc;
        s.ke[2 * c] += 0.5 * kin;
      } else {
        s.U[c] = 0.5f * (s.U_half[c] + Uc);
        s.ke[2 * c + 1] += 0.5 * kin;
        store_key(s.key + 2 * c, k_next);
      }
    } else {
      s.U[c] = Uc;
    }
    if (s.fp8) {
      // delayed scaling: this evaluation's amax sets the next scales; a weight shadow
      // written by this update carries the scale it was written with
      float* qc = s.q + (int64_t)c * kQWords;
      unsigned* am = reinterpret_cast<unsigned*>(qc + 8);
      float a[6], next[2];
#pragma unroll
      for (int t = 0; t < 6; ++t) a[t] = __uint_as_float(am[t]);
      next[0] = qc[6];
      next[1] = qc[7];
#pragma unroll
      for (int t = Q_X; t <= Q_DA1; ++t) {
        if (a[t] > 0.0f) qc[t] = kQTarget / a[t];
        am[t] = 0u;
      }
      if (s.update) {
#pragma unroll
        for (int l = 0; l < 2; ++l) {
          qc[Q_W1 + l] = next[l];
          if (a[Q_W1 + l] > 0.0f) qc[6 + l] = kQTarget / a[Q_W1 + l];
          am[Q_W1 + l] = 0u;
        }
      }
    }
    if (s.update && !obabo) {
      const int ss = s.save_slot ? s.save_slot[it] : -1;
      if (ss >= 0 && ss < s.n_slots && s.samples_U) s.samples_U[(int64_t)c * s.n_slots + ss] = Uc;
      store_key(s.key + 2 * c, k_next);
      store_key(s.dkey + 2 * c, d_next);
      // the last chain advances the iteration counter (read by the next launch)
      const unsigned prev = atomicAdd(s.done, 1u);
      if (prev == (unsigned)s.C - 1) {
        atomicExch(s.done, 0u);
        atomicAdd(s.iter, 1);
      }
    }
  }
}

// Copies theta into the sample buffer at kept iterations (after the step).
__global__ void __launch_bounds__(GT) save_kernel(Step s, int it_offset) {
  const int c = blockIdx.y;
  // the iteration that just completed is iter - 1
  const int it = max(0, min(s.iter[0] - it_offset, s.table_len - 1));
  const int slot = s.save_slot ? s.save_slot[it] : -1;
  if (slot < 0 || slot >= s.n_slots || !s.samples) return;
  for (int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x; i < s.P; i += (int64_t)gridDim.x * GT)
    s.samples[((int64_t)c * s.n_slots + slot) * s.P + i] = s.theta[(int64_t)c * s.P + i];
}

// theta -> bf16 shadow.
__global__ void __launch_bounds__(GT) shadow_kernel(const float* th, uint16_t* sh, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x; i < n; i += (int64_t)gridDim.x * GT)
    sh[i] = f2bf(th[i]);
}

// ------------------------------------------------------------ fp8 set-up ------
__global__ void __launch_bounds__(GT) q_zero_kernel(float* q, int n) {
  const int i = blockIdx.x * GT + threadIdx.x;
  if (i < n) q[i] = 0.0f;
}

// max |W1|, max |W2| of every chain into the amax words.
__global__ void __launch_bounds__(GT) w_amax_kernel(Step s) {
  const int c = blockIdx.y;
  const float* th = s.theta + (int64_t)c * s.P;
  float m0 = 0.f, m1 = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x; i < s.off[2];
       i += (int64_t)gridDim.x * GT) {
    const float a = fabsf(th[i]);
    if (i < s.off[1]) m0 = fmaxf(m0, a);
    else m1 = fmaxf(m1, a);
  }
  q_note_amax(s, c, Q_W1, m0);
  q_note_amax(s, c, Q_W2, m1);
}

// Weight scales from the amax words (current and next shadow), activation scales 1.
__global__ void __launch_bounds__(GT) q_init_kernel(Step s) {
  const int c = blockIdx.x * GT + threadIdx.x;
  if (c >= s.C) return;
  float* qc = s.q + (int64_t)c * kQWords;
  unsigned* am = reinterpret_cast<unsigned*>(qc + 8);
  for (int t = Q_X; t <= Q_DA1; ++t) qc[t] = 1.0f;
  for (int l = 0; l < 2; ++l) {
    const float a = __uint_as_float(am[Q_W1 + l]);
    const float sc = a > 0.0f ? kQTarget / a : 1.0f;
    qc[Q_W1 + l] = sc;
    qc[6 + l] = sc;
    am[Q_W1 + l] = 0u;
  }
}

__global__ void __launch_bounds__(GT) w_quant_kernel(Step s) {
  const int c = blockIdx.y;
  const float* th = s.theta + (int64_t)c * s.P;
  const float* qc = s.q + (int64_t)c * kQWords;
  for (int64_t i = (int64_t)blockIdx.x * GT + threadIdx.x; i < s.off[2];
       i += (int64_t)gridDim.x * GT)
    s.shadow8[(int64_t)c * s.P + i] = f2q(th[i] * qc[i < s.off[1] ? Q_W1 : Q_W2]);
}

// ------------------------------------------------------ full-data potential ----
// out[c] = (-likelihood - log p(theta_c)) / T with the float64 Gaussian log prior; the
// likelihood is facc plus the last chunk's rows. Grid (kFinalBlocks, C), the chain's
// last-arriving block combines the block sums. The parameters are read 16 bytes at a time,
// eight reads in flight (16 chains of 4.2 M, 268 MB: 130 -> 57 us).
__global__ void __launch_bounds__(GT) full_final_kernel(Step s, double* out) {
  __shared__ double red[GT / kWave];
  __shared__ int flag;
  const int c = blockIdx.y;
  double lp = 0.0;
  if (s.has_prior) {
    const double iv = (double)s.prior_inv_var, ln = (double)s.prior_log_norm;
    const float* th = s.theta + (int64_t)c * s.P;
    constexpr int kIn = 8;  // reads in flight
    const int64_t quads = s.P / 4, step = (int64_t)gridDim.x * GT;
    const int64_t t0 = (int64_t)blockIdx.x * GT + threadIdx.x;
    auto add = [&](float wf) __attribute__((always_inline)) {
      const double w = (double)wf;
      lp += (ln + w * w * iv) * -0.5;
    };
    for (int64_t q0 = t0; q0 < quads; q0 += kIn * step) {
      f32x4u x[kIn];
#pragma unroll
      for (int u = 0; u < kIn; ++u)
        x[u] = *reinterpret_cast<const f32x4u*>(th + 4 * min(q0 + u * step, quads - 1));
#pragma unroll
      for (int u = 0; u < kIn; ++u)
        if (q0 + u * step < quads)
#pragma unroll
          for (int e = 0; e < 4; ++e) add(x[u][e]);
    }
    if (4 * quads + t0 < s.P) add(th[4 * quads + t0]);  // the last P % 4
  }
  lp = block_sum_d<GT>(lp, red);
  if (threadIdx.x == 0) publish(s.fin_part + (int64_t)c * gridDim.x + blockIdx.x, lp);
  if (!arrive_last(s.counters + c, gridDim.x, &flag)) return;
  double t = 0.0;
  for (int b = threadIdx.x; b < (int)gridDim.x; b += GT)
    t += consume(s.fin_part + (int64_t)c * gridDim.x + b);
  double lk = 0.0;
  for (int r = threadIdx.x; r < s.n; r += GT) lk += (double)s.lik[(int64_t)c * s.n + r];
  t = block_sum_d<GT>(t, red);
  lk = block_sum_d<GT>(lk, red);
  if (threadIdx.x == 0) out[c] = (-(s.facc[c] + lk) - t) / (double)s.temperature;
}

// ----------------------------------------------------------------- SGGMC MH ----
struct MH {
  double* U_full;
  const double* U_prop;
  float* theta_old;
  float* mom_old;
  float* U_old;
  uint32_t* key;
  float* stats;
  int32_t* accepted;
};

// Every block of chain c evaluates the same decision from inputs that only the chain's
// last-arriving block rewrites, applies it to its slice of the parameters, and saves
// the slice at a kept iteration.
__global__ void __launch_bounds__(GT) mh_kernel(Step s, MH m) {
  __shared__ int flag;
  const int c = blockIdx.y;
  const int it = cur_iter(s);
  const float T = s.noise_temperature;
  const double dE = (m.U_prop[c] - m.U_full[c]) + (s.ke[2 * c + 1] - s.ke[2 * c]);
  double log_alpha = -1.0 / (double)T * dE;
  log_alpha = log_alpha <= 0.0 ? log_alpha : 0.0;
  Key next, sub;
  split2(load_key(m.key + 2 * c), next, sub);
  const float u = bits_to_uniform(bits_word(sub, 1u, 0u), 0.0f, 1.0f);
  const bool accept = (double)logf_cephes(u) < log_alpha;
  const int slot = s.save_slot ? s.save_slot[it] : -1;
  const bool save = s.samples && slot >= 0 && slot < s.n_slots;
  float* th = s.theta + (int64_t)c * s.P;
  float* mo = s.mom + (int64_t)c * s.P;
  float* tho = m.theta_old + (int64_t)c * s.P;
  float* moo = m.mom_old + (int64_t)c * s.P;
  uint16_t* sh = s.fp32 ? nullptr : s.shadow + (int64_t)c * s.P;
  float* smp = save ? s.samples + ((int64_t)c * s.n_slots + slot) * s.P : nullptr;
  auto shadow = [&](int64_t i, float w) __attribute__((always_inline)) {
    if (s.fp8 && i < s.off[2]) {
      const int l = i < s.off[1] ? 0 : 1;
      s.shadow8[(int64_t)c * s.P + i] = f2q(w * s.q[(int64_t)c * kQWords + Q_W1 + l]);
    } else if (!s.fp32) {
      sh[i] = f2bf(w);
    }
  };
  // the kept pair goes from (th, mo) to (tho, moo) or back, 16 bytes at a time, with the
  // reads of four quads in flight (16 chains of 4.2 M, 1.07 GB: 327 -> 229 us)
  const float* ws = accept ? th : tho;
  const float* ms = accept ? mo : moo;
  float* wd = accept ? tho : th;
  float* md = accept ? moo : mo;
  constexpr int kIn = 4;
  const int64_t quads = s.P / 4, step = (int64_t)gridDim.x * GT;
  const int64_t t0 = (int64_t)blockIdx.x * GT + threadIdx.x;
  for (int64_t q0 = t0; q0 < quads; q0 += kIn * step) {
    f32x4u w[kIn], m4[kIn];
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const int64_t i = 4 * min(q0 + u * step, quads - 1);
      w[u] = *reinterpret_cast<const f32x4u*>(ws + i);
      m4[u] = *reinterpret_cast<const f32x4u*>(ms + i);
    }
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const int64_t i = 4 * (q0 + u * step);
      if (i >= 4 * quads) break;
      *reinterpret_cast<f32x4u*>(wd + i) = w[u];
      *reinterpret_cast<f32x4u*>(md + i) = m4[u];
      if (!accept)
#pragma unroll
        for (int e = 0; e < 4; ++e) shadow(i + e, w[u][e]);
      if (save) *reinterpret_cast<f32x4u*>(smp + i) = w[u];
    }
  }
  for (int64_t i = 4 * quads + t0; i < s.P; i += step) {  // the last P % 4
    const float w = ws[i];
    wd[i] = w;
    md[i] = ms[i];
    if (!accept) shadow(i, w);
    if (save) smp[i] = w;
  }
  if (!arrive_last(s.counters + c, gridDim.x, &flag)) return;
  if (threadIdx.x == 0) {
    const float U = accept ? s.U[c] : m.U_old[c];
    s.U[c] = U;
    m.U_old[c] = U;
    if (accept) m.U_full[c] = m.U_prop[c];
    const double dk = s.ke[2 * c + 1] - s.ke[2 * c];
    s.ke[2 * c] = 0.0;
    s.ke[2 * c + 1] = 0.0;
    store_key(m.key + 2 * c, next);
    if (m.accepted && accept) m.accepted[c] += 1;
    if (save && s.samples_U) s.samples_U[(int64_t)c * s.n_slots + slot] = U;
    if (save && m.stats) {
      float* st = m.stats + ((int64_t)c * s.n_slots + slot) * 3;
      st[0] = (float)exp(log_alpha);
      st[1] = s.eps_table[it];
      st[2] = (float)dk;
    }
    const unsigned prev = atomicAdd(s.done, 1u);
    if (prev == (unsigned)s.C - 1) {
      atomicExch(s.done, 0u);
      atomicAdd(s.iter, 1);
    }
  }
}

}  // namespace mlp
}  // namespace sgmc

using namespace sgmc;
using namespace sgmc::mlp;

namespace {

struct Layout {
  int64_t xb, lab, h1, h2, da2, da1, dl, lik, lkey, prior, ke, facc, col, fin, total;
  int nparts, g4_blocks, g5_blocks, small_blocks;
};

int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

Layout layout_of(int C, int n, int D_in, int H1, int H2) {
  Layout L;
  int64_t o = 0;
  // activations sized for float32 elements (the widest precision)
  L.xb = o; o = align256(o + (int64_t)C * n * D_in * 4);
  L.lab = o; o = align256(o + (int64_t)C * n * 4);
  L.h1 = o; o = align256(o + (int64_t)C * n * H1 * 4);
  L.h2 = o; o = align256(o + (int64_t)C * n * H2 * 4);
  L.da2 = o; o = align256(o + (int64_t)C * n * H2 * 4);
  L.da1 = o; o = align256(o + (int64_t)C * n * H1 * 4);
  L.dl = o; o = align256(o + (int64_t)C * n * NCLS * 4);
  L.lik = o; o = align256(o + (int64_t)C * n * 4);
  L.lkey = o; o = align256(o + (int64_t)C * NLEAF * 2 * 4);
  L.g4_blocks = (H1 / BM) * (H2 / BN);
  L.g5_blocks = (D_in / BM) * (H1 / BN);
  const int64_t small_total = (int64_t)H2 * NCLS + H1 + H2 + NCLS;
  L.small_blocks = (int)((small_total + GT - 1) / GT);
  L.nparts = L.g4_blocks + L.g5_blocks + L.small_blocks;
  L.prior = o; o = align256(o + (int64_t)C * L.nparts * 4);
  L.ke = o; o = align256(o + (int64_t)C * L.nparts * 4);
  L.facc = o; o = align256(o + (int64_t)C * 8);
  L.col = o; o = align256(o + (int64_t)C * (n / kStrip) * small_total * 4);
  L.fin = o; o = align256(o + (int64_t)C * kFinalBlocks * 8);
  L.total = o;
  return L;
}

}  // namespace

extern "C" {

int64_t sgmc_mlp_param_count(int D_in, int H1, int H2) {
  return (int64_t)D_in * H1 + (int64_t)H1 * H2 + (int64_t)H2 * NCLS + H1 + H2 + NCLS;
}

int64_t sgmc_mlp_workspace_bytes(int C, int n, int D_in, int H1, int H2) {
  return layout_of(C, n, D_in, H1, H2).total;
}

int sgmc_mlp_shadow(const float* theta, uint16_t* shadow, int64_t count, void* stream) {
  SGMC_REQUIRE(theta && shadow && count >= 0, SGMC_E_ARG, "sgmc_mlp_shadow: bad argument");
  if (count == 0) return SGMC_OK;
  const int64_t blocks = std::min<int64_t>((count + GT - 1) / GT, 65535);
  hipLaunchKernelGGL(shadow_kernel, dim3((unsigned)blocks), dim3(GT), 0, as_stream(stream),
                     theta, shadow, count);
  return check_launch("sgmc_mlp_shadow");
}

}  // extern "C"

namespace {

// Split-K factor of the heuristic; a tuned GEMM may take 4.
constexpr int kMaxSplits = 2;

// Checks tune[] against the shapes: each nonzero entry is 16 k + s with k a k-tile of
// the precision (bf16 32 / 128, e4m3 64 / 128, float32 32), s in {1, 2, 3, 4} (s > 1 for
// the forward GEMMs G1-G3 only) and the GEMM's K a multiple of k s.
int check_tune(int D_in, int H1, int H2, int n, int precision, const int32_t* tune) {
  if (!tune) return SGMC_OK;
  const int K[kSlots] = {D_in, H1, H2, n, n};
  for (int i = 0; i < kSlots; ++i) {
    const int tv = tune[i];
    if (tv == 0) continue;
    const int bk = tv >> 4, sp = tv & 15;
    const bool bk_ok = precision == 2 ? bk == 32 : precision == 1 ? (bk == 64 || bk == 128)
                                                                : (bk == 32 || bk == 128);
    SGMC_REQUIRE(bk_ok && sp >= 1 && sp <= 4 && (sp == 1 || i < SLOT_G4) &&
                     K[i] % (bk * sp) == 0,
                 SGMC_E_ARG, "sgmc_mlp: tune[%d] = %d (k-tile %d, split %d) does not fit K = %d",
                 i, tv, bk, sp, K[i]);
  }
  return SGMC_OK;
}

// The k-tile depth and split-K factor of each GEMM (16 k + s): tune[i] where set, else
// the built-in choice --
// - a k-tile of 128 when K allows (bf16, e4m3), 32 (bf16) or 64 (e4m3) otherwise; 32 for
//   float32 and for the bf16 parameter updates. The k-tile takes part in which splits a
//   code may name; the kernels' stages have one depth.
// - forward GEMMs G1-G3 split K in two while the grid holds at most about four blocks
//   per CU: they have few output tiles but long K. The parameter GEMMs never split. The
//   sums over K follow the split, so it decides last bits and is kept as it is.
void plan_gemms(int D_in, int H1, int H2, int n, int C, int precision, int update,
                const int32_t* tune, int* plan) {
  const int K[kSlots] = {D_in, H1, H2, n, n};
  const int64_t tiles[kSlots] = {(int64_t)(n / BM) * (H1 / BN), (int64_t)(n / BM) * (H2 / BN),
                                 (int64_t)(n / BM) * (H1 / BN), (int64_t)(H1 / BM) * (H2 / BN),
                                 (int64_t)(D_in / BM) * (H1 / BN)};
  for (int i = 0; i < kSlots; ++i) {
    if (tune && tune[i]) {
      plan[i] = tune[i];
      continue;
    }
    int bk;
    if (precision == 2) bk = 32;
    else if (precision == 1) bk = K[i] % 128 == 0 ? 128 : 64;
    else bk = K[i] % 128 == 0 && !(update && i >= SLOT_G4) ? 128 : 32;
    int sp = 1;
    if (i < SLOT_G4) {
      const int64_t blocks = tiles[i] * C;
      const int ktiles = K[i] / bk;
      while (sp < kMaxSplits && blocks * sp * 2 <= 1024 && ktiles % (sp * 2) == 0) sp *= 2;
    }
    plan[i] = bk * 16 + sp;
  }
}

// Operand / output formats and scale slots of one GEMM.
Gemm with_q(Gemm g, int ta, int tb, int tout) {
  g.ta = ta;
  g.tb = tb;
  g.tout = tout;
  return g;
}

// Validates the state and fills the kernels' view of it.
int make_step(const sgmc_mlp_state* st, int update, Layout& L, Step& s) {
  SGMC_REQUIRE(st, SGMC_E_ARG, "sgmc_mlp: null state");
  const sgmc_mlp_state& q = *st;
  SGMC_REQUIRE(q.precision >= 0 && q.precision <= 2, SGMC_E_ARG,
               "sgmc_mlp: precision %d is not 0 (bf16), 1 (fp8) or 2 (fp32)", q.precision);
  SGMC_REQUIRE(q.X && q.labels && q.theta && (q.shadow || q.precision == 2) && q.key &&
                   q.dkey && q.work && q.U &&
                   q.eps_table && q.iter && q.counters && q.done,
               SGMC_E_ARG, "sgmc_mlp: null pointer in state");
  SGMC_REQUIRE(update || q.grad, SGMC_E_ARG, "sgmc_mlp_step: gradient mode needs grad");
  SGMC_REQUIRE(q.C >= 1 && q.n >= 1 && q.N >= 1 && q.N <= 2147483647LL, SGMC_E_ARG,
               "sgmc_mlp: bad C/n/N");
  SGMC_REQUIRE(q.n % BM == 0 && q.D_in % BM == 0 && q.H1 % BM == 0, SGMC_E_ARG,
               "sgmc_mlp: n, D_in and H1 must be multiples of %d", BM);
  SGMC_REQUIRE(q.H1 % BN == 0 && q.H2 % BN == 0, SGMC_E_ARG,
               "sgmc_mlp: H1 and H2 must be multiples of %d", BN);
  SGMC_REQUIRE(q.ldx % 4 == 0 && q.ldx >= q.D_in && ((uintptr_t)q.X & 15) == 0, SGMC_E_ARG,
               "sgmc_mlp: X rows must be 16-byte aligned with ldx %% 4 == 0");
  SGMC_REQUIRE(q.P == sgmc_mlp_param_count(q.D_in, q.H1, q.H2), SGMC_E_ARG,
               "sgmc_mlp: P does not match the layer sizes");
  SGMC_REQUIRE(q.table_len >= 1 && q.temperature != 0.0f, SGMC_E_ARG,
               "sgmc_mlp: bad schedule");
  SGMC_REQUIRE((int64_t)q.D_in * q.H1 < 4294967295LL, SGMC_E_ARG, "sgmc_mlp: W1 too large");
  SGMC_REQUIRE(q.mode >= MLP_SGLD && q.mode <= MLP_OBABO_BO, SGMC_E_ARG, "sgmc_mlp: bad mode");
  if (update && q.mode != MLP_SGLD)
    SGMC_REQUIRE(q.mom && q.ke && q.U_half && q.decay_table && q.noise_table, SGMC_E_ARG,
                 "sgmc_mlp_step: OBABO needs mom, ke, U_half and the decay / noise tables");
  L = layout_of(q.C, q.n, q.D_in, q.H1, q.H2);
  SGMC_REQUIRE(q.work_bytes >= L.total, SGMC_E_ARG, "sgmc_mlp: workspace too small");
  uint8_t* w = static_cast<uint8_t*>(q.work);
  s.X = q.X; s.labels = q.labels; s.N = q.N; s.ldx = q.ldx;
  s.D_in = q.D_in; s.H1 = q.H1; s.H2 = q.H2; s.n = q.n; s.C = q.C;
  s.theta = q.theta; s.v = q.rms ? q.v : nullptr; s.shadow = q.shadow; s.P = q.P;
  const int64_t sizes[NLEAF] = {(int64_t)q.D_in * q.H1, (int64_t)q.H1 * q.H2,
                                (int64_t)q.H2 * NCLS, q.H1, q.H2, NCLS};
  int64_t o = 0;
  for (int l = 0; l < NLEAF; ++l) {
    s.off[l] = o;
    s.size[l] = sizes[l];
    o += sizes[l];
  }
  s.key = q.key; s.dkey = q.dkey;
  s.rmult = randint_mult((uint32_t)q.N);
  s.rmagic = randint_magic((uint32_t)q.N);
  s.Xb = w + L.xb;
  s.lab = reinterpret_cast<int32_t*>(w + L.lab);
  s.h1 = w + L.h1;
  s.h2 = w + L.h2;
  s.da2 = w + L.da2;
  s.da1 = w + L.da1;
  s.dL = reinterpret_cast<float*>(w + L.dl);
  s.lik = reinterpret_cast<float*>(w + L.lik);
  s.lkey = reinterpret_cast<uint32_t*>(w + L.lkey);
  s.prior_part = reinterpret_cast<float*>(w + L.prior);
  s.ke_part = reinterpret_cast<float*>(w + L.ke);
  s.col_part = reinterpret_cast<float*>(w + L.col);
  s.fin_part = reinterpret_cast<double*>(w + L.fin);
  s.facc = reinterpret_cast<double*>(w + L.facc);
  s.nparts = L.nparts;
  s.U = q.U; s.grad = q.grad;
  s.samples = q.samples; s.samples_U = q.samples_U; s.n_slots = q.n_slots;
  s.eps_table = q.eps_table; s.save_slot = q.save_slot; s.iter = q.iter;
  s.counters = q.counters; s.done = q.done; s.table_len = q.table_len;
  s.rms = q.rms && q.v ? 1 : 0;
  s.update = update ? 1 : 0;
  s.alpha = q.alpha; s.lmbd = q.lmbd; s.temperature = q.temperature;
  s.noise_temperature = q.noise_temperature;
  s.has_prior = q.has_prior;
  const float ps2 = q.prior_scale * q.prior_scale;
  s.prior_inv_var = q.has_prior ? 1.0f / ps2 : 0.0f;
  s.prior_log_norm = q.has_prior ? logf(2.0f * (float)M_PI * ps2) : 0.0f;
  s.mode = update ? q.mode : MLP_SGLD;
  s.mom = q.mom; s.ke = q.ke; s.U_half = q.U_half;
  s.decay_table = q.decay_table; s.noise_table = q.noise_table;
  s.full = 0;
  s.row0 = 0;
  s.fp8 = q.precision == 1 ? 1 : 0;
  s.fp32 = q.precision == 2 ? 1 : 0;
  const int trc = check_tune(q.D_in, q.H1, q.H2, q.n, q.precision, q.tune);
  if (trc != SGMC_OK) return trc;
  int plan[kSlots];
  plan_gemms(q.D_in, q.H1, q.H2, q.n, q.C, q.precision, update, q.tune, plan);
  for (int i = SLOT_G1; i <= SLOT_G3; ++i) s.split[i] = plan[i] & 15;
  s.q = q.q;
  s.shadow8 = q.shadow8;
  if (s.fp8)
    SGMC_REQUIRE(q.q && q.shadow8, SGMC_E_ARG, "sgmc_mlp: fp8 precision needs q and shadow8");
  return SGMC_OK;
}

// GEMM operand of weight leaf l (W1, W2): the e4m3 or bf16 shadow, or theta itself.
const void* gemm_weight(const Step& s, const sgmc_mlp_state& q, int l) {
  if (s.fp32) return q.theta + s.off[l];
  if (s.fp8) return q.shadow8 + s.off[l];
  return q.shadow + s.off[l];
}

template <int PREC, int R, int NW>
void launch_head_as(const Step& s, hipStream_t st) {
  const size_t lds = (size_t)s.H2 * kW3Stride * sizeof(float);
  const dim3 grid(s.n / (R * NW), s.C), block(kWave * NW);
  if (lds <= 65536) hipLaunchKernelGGL((head_kernel<PREC, true, R, NW>), grid, block, lds, st, s);
  else hipLaunchKernelGGL((head_kernel<PREC, false, R, NW>), grid, block, 0, st, s);
}
// Rows per wavefront and wavefronts per block: as many rows as still give every CU two
// blocks of eight wavefronts (a block stages W3 once, a read of a W3 row serves all rows of
// the wavefront), one row and four wavefronts when there are few. Measured, us per launch:
// 8192 rows of H2 = 1024 (98 full passes and 20 evaluations): 4 x 8 13.1, 4 x 4 15.3,
// 2 x 8 14.7, 2 x 4 21.5; 4096 rows of H2 = 512: 2 x 8 9.7, 2 x 4 11.1, 1 x 8 10.7,
// 1 x 4 12.2.
template <int PREC>
void launch_head_by(const Step& s, hipStream_t st) {
  const int64_t rows = (int64_t)s.C * s.n;
  if (rows >= 8192) launch_head_as<PREC, 4, 8>(s, st);
  else if (rows >= 4096) launch_head_as<PREC, 2, 8>(s, st);
  else launch_head_as<PREC, 1, 4>(s, st);
}

// The head over rows [0, n) of every chain.
void launch_head(const Step& s, hipStream_t st) {
  if (s.fp32) launch_head_by<P_F32>(s, st);
  else if (s.fp8) launch_head_by<P_FP8>(s, st);
  else launch_head_by<P_BF16>(s, st);
}

// gather, forward GEMMs and the head (likelihood, and its backward unless s.full).
void launch_forward(const Step& s, const sgmc_mlp_state& q, hipStream_t st_) {
  const int C = q.C, n = q.n;
  // eight rows per block share a draw and an atomic; two while eight would leave CUs without
  // a block (4 x 256 rows: 9.9 us for 11.7)
  if (s.full)
    hipLaunchKernelGGL((gather_kernel<true, 8>),
                       dim3(n / 8, (C + kGatherChains - 1) / kGatherChains), dim3(8 * kWave), 0,
                       st_, s);
  else if ((int64_t)C * n >= 4096)
    hipLaunchKernelGGL((gather_kernel<false, 8>), dim3(n / 8, C), dim3(8 * kWave), 0, st_, s);
  else
    hipLaunchKernelGGL((gather_kernel<false, 2>), dim3(n / 2, C), dim3(2 * kWave), 0, st_, s);
  const void* W1 = gemm_weight(s, q, 0);
  const void* W2 = gemm_weight(s, q, 1);
  Gemm g1{s.Xb, q.D_in, (int64_t)n * q.D_in, W1, q.H1, q.P, n, q.H1, q.D_in,
          s.h1, q.H1, (int64_t)n * q.H1, q.theta + s.off[3], q.P, nullptr, 0, 0, 0, 0};
  launch_act_gemm(with_q(g1, Q_X, Q_W1, Q_H1), s, st_, s.split[SLOT_G1]);
  Gemm g2{s.h1, q.H1, (int64_t)n * q.H1, W2, q.H2, q.P, n, q.H2, q.H1,
          s.h2, q.H2, (int64_t)n * q.H2, q.theta + s.off[4], q.P, nullptr, 0, 0, 0, 0};
  launch_act_gemm(with_q(g2, Q_H1, Q_W2, -1), s, st_, s.split[SLOT_G2]);
  launch_head(s, st_);
}

}  // namespace

extern "C" {

int sgmc_mlp_gemm_plan(int D_in, int H1, int H2, int n, int C, int precision, int update,
                       const int32_t* tune, int32_t* plan) {
  SGMC_REQUIRE(plan && C >= 1 && n >= BM && n % BM == 0 && D_in % BM == 0 && H1 % BN == 0 &&
                   H2 % BN == 0 && precision >= 0 && precision <= 2,
               SGMC_E_ARG, "sgmc_mlp_gemm_plan: bad shape or precision");
  const int rc = check_tune(D_in, H1, H2, n, precision, tune);
  if (rc != SGMC_OK) return rc;
  int p[kSlots];
  plan_gemms(D_in, H1, H2, n, C, precision, update, tune, p);
  for (int i = 0; i < kSlots; ++i) plan[i] = p[i];
  return SGMC_OK;
}

int sgmc_mlp_step(const sgmc_mlp_state* st, int update, void* stream) {
  Layout L;
  Step s;
  const int rc = make_step(st, update, L, s);
  if (rc != SGMC_OK) return rc;
  const sgmc_mlp_state& q = *st;
  hipStream_t st_ = as_stream(stream);
  const int C = q.C, n = q.n;
  launch_forward(s, q, st_);
  const void* W2 = gemm_weight(s, q, 1);
  // dA1 = (dA2 W2^T) * (H1 > 0): B[k=b][n=a] = W2[a][b], k-contiguous rows of W2.
  Gemm g3{s.da2, q.H2, (int64_t)n * q.H2, W2, q.H2, q.P, n, q.H1, q.H2,
          s.da1, q.H1, (int64_t)n * q.H1, nullptr, 0, s.h1, q.H1, (int64_t)n * q.H1, 0, 0};
  launch_act_gemm(with_q(g3, Q_DA2, Q_W2, Q_DA1), s, st_, s.split[SLOT_G3]);
  // gW2 = H1^T dA2: A[m=a][k=i] = H1[i][a] (m-contiguous), B[k=i][n=b] = dA2[i][b].
  Gemm g4{s.h1, q.H1, (int64_t)n * q.H1, s.da2, q.H2, (int64_t)n * q.H2, q.H1, q.H2, n,
          nullptr, 0, 0, nullptr, 0, nullptr, 0, 0, 1, 0};
  // gW1 = Xb^T dA1.
  Gemm g5{s.Xb, q.D_in, (int64_t)n * q.D_in, s.da1, q.H1, (int64_t)n * q.H1, q.D_in, q.H1, n,
          nullptr, 0, 0, nullptr, 0, nullptr, 0, 0, 0, L.g4_blocks};
  g4 = with_q(g4, Q_H1, Q_DA2, -1);
  g5 = with_q(g5, Q_X, Q_DA1, -1);
  launch_param_gemms(g4, g5, s, st_);  // and the strips' column sums
  hipLaunchKernelGGL(small_kernel, dim3(L.small_blocks, C), dim3(GT), 0, st_, s,
                     L.g4_blocks + L.g5_blocks);
  if (update && s.mode == MLP_SGLD && q.samples && q.save_slot) {
    hipLaunchKernelGGL(save_kernel, dim3(256, C), dim3(GT), 0, st_, s, 1);
  }
  return check_launch("sgmc_mlp_step");
}

int sgmc_mlp_init_fp8(const sgmc_mlp_state* st, void* stream) {
  Layout L;
  Step s;
  const int rc = make_step(st, 1, L, s);
  if (rc != SGMC_OK) return rc;
  SGMC_REQUIRE(s.fp8, SGMC_E_ARG, "sgmc_mlp_init_fp8: state precision is not fp8");
  hipStream_t st_ = as_stream(stream);
  const int nq = st->C * kQWords;
  hipLaunchKernelGGL(q_zero_kernel, dim3((nq + GT - 1) / GT), dim3(GT), 0, st_, s.q, nq);
  hipLaunchKernelGGL(w_amax_kernel, dim3(512, st->C), dim3(GT), 0, st_, s);
  hipLaunchKernelGGL(q_init_kernel, dim3((st->C + GT - 1) / GT), dim3(GT), 0, st_, s);
  hipLaunchKernelGGL(w_quant_kernel, dim3(512, st->C), dim3(GT), 0, st_, s);
  return check_launch("sgmc_mlp_init_fp8");
}

int sgmc_mlp_full_potential(const sgmc_mlp_state* st, double* out, void* stream) {
  Layout L;
  Step s;
  const int rc = make_step(st, 1, L, s);
  if (rc != SGMC_OK) return rc;
  SGMC_REQUIRE(out, SGMC_E_ARG, "sgmc_mlp_full_potential: null output");
  const sgmc_mlp_state& q = *st;
  hipStream_t st_ = as_stream(stream);
  s.full = 1;
  for (int64_t r0 = 0; r0 < q.N; r0 += q.n) {
    s.row0 = r0;
    launch_forward(s, q, st_);
  }
  hipLaunchKernelGGL(full_final_kernel, dim3(kFinalBlocks, q.C), dim3(GT), 0, st_, s, out);
  return check_launch("sgmc_mlp_full_potential");
}

int sgmc_mlp_mh(const sgmc_mlp_state* st, void* stream) {
  Layout L;
  Step s;
  const int rc = make_step(st, 1, L, s);
  if (rc != SGMC_OK) return rc;
  const sgmc_mlp_state& q = *st;
  SGMC_REQUIRE(q.mom && q.ke && q.U_full && q.U_prop && q.theta_old && q.mom_old && q.U_old &&
                   q.mh_key,
               SGMC_E_ARG, "sgmc_mlp_mh: null pointer in state");
  SGMC_REQUIRE(q.noise_temperature != 0.0f, SGMC_E_ARG, "sgmc_mlp_mh: zero temperature");
  s.mom = q.mom;
  s.ke = q.ke;
  MH m{q.U_full, q.U_prop, q.theta_old, q.mom_old, q.U_old, q.mh_key, q.mh_stats, q.accepted};
  const int64_t blocks = std::min<int64_t>((q.P + 16 * GT - 1) / (16 * GT), 1024);
  hipLaunchKernelGGL(mh_kernel, dim3((unsigned)blocks, q.C), dim3(GT), 0, as_stream(stream), s,
                     m);
  return check_launch("sgmc_mlp_mh");
}

}  // extern "C"
