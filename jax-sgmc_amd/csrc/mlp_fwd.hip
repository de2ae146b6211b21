// The activation GEMMs of the MLP engine: H1 = relu(Xb W1 + b1), H2 = relu(H1 W2 + b2) and
// dA1 = (dA2 W2^T) * (H1 > 0), one launch each.
//
// What bounds them: the operand traffic into the CUs. Xb W1 of a 3072-512 net (16 chains,
// n = 256, bf16) is 13 GFLOP on 75 MB, but every CU pulls 1.2 MB through its 32 KB cache,
// whose outstanding lines at the latency of HBM give about 15 bytes per cycle: 38 us, the
// matrix cores 15% busy. Deeper register prefetch and padded row strides change nothing. A block of G groups computes a TM x TN tile of one chain, every group a
// G-th of K: the K halves of a split GEMM meet in LDS instead of in a partial-product array
// and a second launch. Operands go through LDS in stages of 128 bytes of k per row, two
// stages deep in registers and two in LDS, one barrier per stage. B with n-contiguous rows
// (the weights as they lie in theta) is staged as it is and read with the transposing LDS
// loads: transposing 8x8 blocks in registers kept the vector ALU busier than the matrix
// cores. Against register transposes, one stage and a partial-product array: 16 chains of
// 3072-512-512 in bf16, the three GEMMs 83 -> 50 us (7 of them by the gather's loads); 3072-1024-1024 in e4m3, n = 512,
// 138 -> 90 us; 4 chains of 3072-512-512 in float32 105 -> 62 us. The k order of the matrix instructions and of the sum over the groups does not
// depend on the tile, so neither do the results.
#include "mlp_tile.h"

namespace sgmc {
namespace mlp {
namespace {

// Four consecutive mask elements, loaded as they lie.
template <int PREC>
struct Mask4 {
  uint8_t b[4 * elem_bytes<PREC>()];
};

// WM x WN wavefronts per group over the TM x TN tile; G groups over K.
template <int PREC, int TM, int TN, int WM, int WN, int G, bool B_K, int EPI>
__global__ void __launch_bounds__(kWave* WM* WN* G) fwd_kernel(Gemm g, Step s, uint32_t gx,
                                                               uint32_t gy) {
  constexpr bool F8 = PREC == P_FP8, f32 = PREC == P_F32;
  constexpr int EB = elem_bytes<PREC>();
  constexpr int NT = kWave * WM * WN;          // threads per group
  constexpr int KE = kStage / EB;              // k-values per stage
  constexpr int kBuf = (TM + TN) * kStage;     // bytes of one stage
  constexpr int kTile = TM * TN * 4;           // bytes of one group's product
  constexpr int MI = TM / WM / 32, NI = TN / WN / 32;
  constexpr int kLds = G * (2 * kBuf > kTile ? 2 * kBuf : kTile);
  static_assert(MI >= 1 && NI >= 1 && kLds <= 160 * 1024, "tile shape");
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  __shared__ float red[WM * WN * G];

  // XCD x takes the contiguous range [x T / 8, (x + 1) T / 8) of tiles (m fastest, then n,
  // then chain), so the blocks that share an operand read it through one L2
  const uint32_t T = gridDim.x;
  uint32_t lin = blockIdx.x;
  if (T % kXcds == 0) lin = (lin % kXcds) * (T / kXcds) + lin / kXcds;
  const int bm = (int)(lin % gx), bn = (int)((lin / gx) % gy), c = (int)(lin / (gx * gy));
  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
  const int t = (int)threadIdx.x % NT;
  const int lane = t & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const int m0 = (w % WM) * (TM / WM), n0 = (w / WM) * (TN / WN);

  const int kspan = g.K / G, kfirst = grp * kspan;
  const uint32_t lda = (uint32_t)(g.lda * EB), ldb = (uint32_t)(g.ldb * EB);
  typedef Stage<PREC, TM, NT, true> StageA;
  typedef Stage<PREC, TN, NT, B_K> StageB;
  const uint8_t* A = reinterpret_cast<const uint8_t*>(g.A) + (int64_t)c * g.sA * EB +
                     (int64_t)(bm * TM + StageA::first(t)) * lda + (int64_t)kfirst * EB;
  const uint8_t* B = reinterpret_cast<const uint8_t*>(g.B) + (int64_t)c * g.sB * EB +
                     (B_K ? (int64_t)(bn * TN + StageB::first(t)) * ldb + (int64_t)kfirst * EB
                          : (int64_t)kfirst * ldb + (int64_t)(bn * TN) * EB);
  const int stages = (kspan + KE - 1) / KE;
  const int64_t stepB = B_K ? (int64_t)kStage : (int64_t)KE * ldb;

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  StageA pa, qa;
  StageB pb, qb;
  auto load = [&](auto& a, auto& b, int st) __attribute__((always_inline)) {
    a.load(A + (int64_t)st * kStage, lda, kspan - st * KE, t);
    b.load(B + st * stepB, ldb, kspan - st * KE, t);
    __builtin_amdgcn_sched_barrier(0);  // stages stay in issue order
  };
  uint8_t* const buf0 = lds + grp * (kLds / G);
  uint8_t* const buf1 = buf0 + kBuf;
  auto put = [&](const auto& a, const auto& b, uint8_t* buf) __attribute__((always_inline)) {
    a.store(buf, t);
    b.store(buf + TM * kStage, t);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](const uint8_t* buf) __attribute__((always_inline)) {
    const uint8_t* As = buf;
    const uint8_t* Bs = buf + TM * kStage;
#pragma unroll
    for (int kk = 0; kk < KE; kk += k_span<PREC>()) {
      typename FragOf<PREC>::T a[MI], b[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) a[i] = frag_k<PREC>(As, m0 + 32 * i, kk, lane);
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        if constexpr (B_K) b[j] = frag_k<PREC>(Bs, n0 + 32 * j, kk, lane);
        else b[j] = frag_n<PREC, TN>(Bs, n0 + 32 * j, kk, lane);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) mma<PREC>(acc[i][j], a[i], b[j]);
    }
  };

  load(pa, pb, 0);
  load(qa, qb, 1);
  put(pa, pb, buf0);
  load(pa, pb, 2);
  lds_sync();
  // (an odd number of stages multiplies one of zeros at the end: a loop of whole pairs
  // without exits keeps the waits exact)
  for (int st = 0; st < stages; st += 2) {
    multiply(buf0);
    put(qa, qb, buf1);
    load(qa, qb, st + 3);
    lds_sync();
    multiply(buf1);
    put(pa, pb, buf0);
    load(pa, pb, st + 4);
    lds_sync();
  }

  // Epilogue: the products meet in LDS (four consecutive columns per lane and write, their
  // position in the row swizzled by m) and are read back row by row, so masks and outputs
  // are whole lines.
  constexpr int kQuads = TN / 4;
  const bool q8 = F8 && g.tout >= 0;
  const float* qc = F8 ? s.q + (int64_t)c * kQWords : nullptr;
  const float ab = F8 ? 1.0f / (qc[g.ta] * qc[g.tb]) : 1.0f;
  const float qs = q8 ? qc[g.tout] : 1.0f;
  const int qd = (int)threadIdx.x % kQuads, r0 = (int)threadIdx.x / kQuads;
  constexpr int kRows = NT * G / kQuads;  // rows per pass
  constexpr int kIts = (TM + kRows - 1) / kRows;
  static_assert(NT * G % kQuads == 0, "readout passes");
  const int col = bn * TN + 4 * qd;
  Mask4<PREC> mk[EPI == EPI_MASK ? kIts : 1];
  if constexpr (EPI == EPI_MASK) {
    const uint8_t* mp = reinterpret_cast<const uint8_t*>(g.mask) +
                        ((int64_t)c * g.sM + (int64_t)(bm * TM) * g.ldm + col) * EB;
#pragma unroll
    for (int i = 0; i < kIts; ++i) {
      const int m = min(r0 + i * kRows, TM - 1);
      __builtin_memcpy(&mk[i], __builtin_assume_aligned(mp + (int64_t)m * g.ldm * EB, 4 * EB),
                       4 * EB);
    }
  }
  f32x4 bias{0.f, 0.f, 0.f, 0.f};
  if constexpr (EPI == EPI_BIAS_RELU)
    bias = *reinterpret_cast<const f32x4u*>(g.bias + (int64_t)c * g.sBias + col);
  float* const prod = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + 32 * i + (lane & 31);
    float* row = prod + grp * (TM * TN) + m * TN;
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = (n0 + 32 * j + 8 * e) / 4 + (lane >> 5);
        *reinterpret_cast<f32x4*>(row + 4 * (q ^ (m & (kQuads - 1)))) =
            f32x4{acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2],
                  acc[i][j][4 * e + 3]};
      }
  }
  lds_sync();
  uint8_t* out = reinterpret_cast<uint8_t*>(g.out) + (int64_t)c * g.sO * act_bytes(q8, f32);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kIts; ++i) {
    const int m = r0 + i * kRows;
    if (TM % kRows != 0 && m >= TM) break;
    const float* p = prod + m * TN + 4 * (qd ^ (m & (kQuads - 1)));
    f32x4 a{0.f, 0.f, 0.f, 0.f};
    if constexpr (G == 1) {
      a = *reinterpret_cast<const f32x4*>(p);
    } else {
#pragma unroll
      for (int v = 0; v < G; ++v) {
        const f32x4 pv = *reinterpret_cast<const f32x4*>(p + v * (TM * TN));
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] += pv[u];
      }
    }
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float r = ab * a[u];
      if constexpr (EPI == EPI_BIAS_RELU) v[u] = fmaxf(r + bias[u], 0.0f);
      else v[u] = mask_on<PREC>(mk[i].b, u) ? r : 0.0f;
      amax = fmaxf(amax, fabsf(v[u]));
    }
    const int64_t o = (int64_t)(bm * TM + m) * g.ldo + col;
    if constexpr (f32) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + o) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
      if (q8) {
        *reinterpret_cast<uint32_t*>(out + o) =
            (uint32_t)f2q(v[0] * qs) | ((uint32_t)f2q(v[1] * qs) << 8) |
            ((uint32_t)f2q(v[2] * qs) << 16) | ((uint32_t)f2q(v[3] * qs) << 24);
      } else {
        *reinterpret_cast<uint2*>(out + 2 * o) =
            make_uint2((uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                       (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
      }
    }
  }
  if (q8) q_note_amax_block(s, c, g.tout, amax, red);
}

template <int PREC, int TM, int TN, int WM, int WN, int G, bool B_K, int EPI>
void launch(const Gemm& g, const Step& s, hipStream_t st) {
  const uint32_t gx = (uint32_t)(g.M / TM), gy = (uint32_t)(g.N / TN);
  hipLaunchKernelGGL((fwd_kernel<PREC, TM, TN, WM, WN, G, B_K, EPI>),
                     dim3(gx * gy * (uint32_t)s.C), dim3(kWave * WM * WN * G), 0, st, g, s, gx, gy);
}

// Tile of a GEMM: the largest that still gives every CU a block (one resident block of 96 or
// 128 KB, two of 64 KB), since a tile's operand traffic per output falls with its edges.
// Measured, Xb W1 and H1 W2 of 16 chains together: e4m3 3072-1024-1024, n = 512, one group:
// 256 x 128 (256 blocks) 66 us, 128 x 128 (512 blocks) 71 us, 64 x 128 82 us; bf16
// 3072-512-512, n = 256, two groups: 64 x 128 (256 blocks) 47 us, 64 x 64 54 us. Float32 is
// bound by the matrix cores, and at few tiles by the number of SIMDs that have one: 32 x 64
// tiles at 4 chains take 52 us where one group per K half in launches of their own took
// 81 us.
template <int PREC, bool B_K, int EPI>
void dispatch(const Gemm& g, const Step& s, hipStream_t st, int splits) {
  const int64_t blocks = (int64_t)(g.M / 64) * (g.N / 128) * s.C;  // of 64 x 128
  if (splits == 1) {
    if (g.M % 256 == 0 && blocks >= 1024) launch<PREC, 256, 128, 4, 2, 1, B_K, EPI>(g, s, st);
    else if (g.M % 128 == 0 && blocks >= 1024) launch<PREC, 128, 128, 2, 2, 1, B_K, EPI>(g, s, st);
    else if (blocks >= 256) launch<PREC, 64, 128, 2, 2, 1, B_K, EPI>(g, s, st);
    else launch<PREC, 64, 64, 2, 2, 1, B_K, EPI>(g, s, st);
  } else if (splits == 2) {
    if (blocks >= 256) launch<PREC, 64, 128, 2, 2, 2, B_K, EPI>(g, s, st);
    else if (PREC == P_F32) launch<PREC, 32, 64, 1, 2, 2, B_K, EPI>(g, s, st);
    else launch<PREC, 64, 64, 2, 2, 2, B_K, EPI>(g, s, st);
  } else if (splits == 3) {
    launch<PREC, 32, 64, 1, 2, 3, B_K, EPI>(g, s, st);
  } else {
    launch<PREC, 32, 64, 1, 2, 4, B_K, EPI>(g, s, st);
  }
}

template <bool B_K, int EPI>
void by_precision(const Gemm& g, const Step& s, hipStream_t st, int splits) {
  if (s.fp32) dispatch<P_F32, B_K, EPI>(g, s, st, splits);
  else if (s.fp8) dispatch<P_FP8, B_K, EPI>(g, s, st, splits);
  else dispatch<P_BF16, B_K, EPI>(g, s, st, splits);
}

}  // namespace

void launch_act_gemm(const Gemm& g, const Step& s, hipStream_t st, int splits) {
  if (g.mask) by_precision<true, EPI_MASK>(g, s, st, splits);
  else by_precision<false, EPI_BIAS_RELU>(g, s, st, splits);
}

}  // namespace mlp
}  // namespace sgmc
