// Column sums of the MLP's small leaves, run as blocks of the parameter GEMMs' launch.
#pragma once
#include "mlp_common.h"

namespace sgmc {
namespace mlp {

// Element i of an activation tensor stored at precision PREC (e4m3 at scale qs).
template <int PREC>
__device__ __forceinline__ float act_of(const void* p, int64_t i, float qs) {
  if constexpr (PREC == P_F32) return reinterpret_cast<const float*>(p)[i];
  else if constexpr (PREC == P_FP8) return q2f(reinterpret_cast<const uint8_t*>(p)[i]) / qs;
  else return bf2f(reinterpret_cast<const uint16_t*>(p)[i]);
}

// Row-strip partial sums of the small leaves' gradients (flat order W3 [H2][10], b1,
// b2, b3): for strip t, part[t][.] = sum over its kStrip rows of h2^T dL, dA1, dA2, dL.
// Block bx of a strip: ceil(H2 / GT) for W3 and b2, ceil(H1 / GT) for b1, one for b3.
// PREC: the evaluation's GEMM precision (h2 is bf16 in e4m3 mode). A thread loads its
// column's kStrip rows before summing them (in ascending row order), one memory round
// trip per strip; the strip's dL rows are staged in LDS.
template <int PREC>
__device__ __forceinline__ void colsum_block(const Step& s, int bx, int t, int c, float* dls) {
  constexpr int H2P = PREC == P_F32 ? P_F32 : P_BF16;
  const int nb2 = (s.H2 + GT - 1) / GT, nb1 = (s.H1 + GT - 1) / GT;
  const int64_t nW3 = (int64_t)s.H2 * NCLS;
  const int64_t total = nW3 + s.H1 + s.H2 + NCLS;
  float* out = s.col_part + ((int64_t)c * (s.n / kStrip) + t) * total;
  const int64_t r0 = (int64_t)c * s.n + (int64_t)t * kStrip;
  const float* dL = s.dL + r0 * NCLS;
  if (bx < nb2) {
    for (int q = threadIdx.x; q < kStrip * NCLS; q += GT) dls[q] = dL[q];
    __syncthreads();
    const int a = bx * GT + threadIdx.x;
    if (a >= s.H2) return;
    const float qs = PREC == P_FP8 ? s.q[(int64_t)c * kQWords + Q_DA2] : 1.0f;
    float h[kStrip], d2[kStrip];
#pragma unroll
    for (int r = 0; r < kStrip; ++r) {
      h[r] = act_of<H2P>(s.h2, (r0 + r) * s.H2 + a, 1.0f);
      d2[r] = act_of<PREC>(s.da2, (r0 + r) * s.H2 + a, qs);
    }
    float w3[NCLS];
#pragma unroll
    for (int k = 0; k < NCLS; ++k) w3[k] = 0.f;
    float b2 = 0.f;
#pragma unroll
    for (int r = 0; r < kStrip; ++r) {
      b2 += d2[r];
#pragma unroll
      for (int k = 0; k < NCLS; ++k) w3[k] += h[r] * dls[r * NCLS + k];
    }
#pragma unroll
    for (int k = 0; k < NCLS; ++k) out[(int64_t)a * NCLS + k] = w3[k];
    out[nW3 + s.H1 + a] = b2;
  } else if (bx < nb2 + nb1) {
    const int i = (bx - nb2) * GT + threadIdx.x;
    if (i >= s.H1) return;
    const float qs = PREC == P_FP8 ? s.q[(int64_t)c * kQWords + Q_DA1] : 1.0f;
    float d1[kStrip];
#pragma unroll
    for (int r = 0; r < kStrip; ++r) d1[r] = act_of<PREC>(s.da1, (r0 + r) * s.H1 + i, qs);
    float b1 = 0.f;
#pragma unroll
    for (int r = 0; r < kStrip; ++r) b1 += d1[r];
    out[nW3 + i] = b1;
  } else {
    const int k = threadIdx.x;
    if (k >= NCLS) return;
    float dk[kStrip];
#pragma unroll
    for (int r = 0; r < kStrip; ++r) dk[r] = dL[r * NCLS + k];
    float b3 = 0.f;
#pragma unroll
    for (int r = 0; r < kStrip; ++r) b3 += dk[r];
    out[nW3 + s.H1 + s.H2 + k] = b3;
  }
}

// Blocks in x of one strip.
inline int colsum_blocks(const Step& s) { return (s.H2 + GT - 1) / GT + (s.H1 + GT - 1) / GT + 1; }

}  // namespace mlp
}  // namespace sgmc
