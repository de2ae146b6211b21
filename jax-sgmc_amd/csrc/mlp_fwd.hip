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
// 3072-512-512 in bf16, the three GEMMs 83 -> 57 us; 3072-1024-1024 in e4m3, n = 512,
// 138 -> 95 us; 4 chains of 3072-512-512 in float32 105 -> 62 us. The k order of the matrix instructions and of the sum over the groups does not
// depend on the tile, so neither do the results.
#include "mlp_common.h"

namespace sgmc {
namespace mlp {
namespace {

constexpr int kStage = 128;  // bytes of k per row and stage

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// k-values of one multiply step: one 32x32x16 instruction, or four 32x32x2 (float32).
template <int PREC>
constexpr int k_span() {
  return PREC == P_F32 ? 8 : 16;
}

// 16-byte chunk swizzle of row r of a k-contiguous tile (8 chunks per row): the fragment
// reads of 32 consecutive rows spread over the banks.
__device__ __forceinline__ int swz_k(int r) { return (r ^ (r >> 3)) & 7; }

// Chunk swizzle of k-row r of an n-contiguous tile of TN columns: the rows that one
// transposing read of a wavefront touches lie in different banks.
template <int PREC, int TN>
__device__ __forceinline__ int swz_n(int r) {
  if constexpr (PREC == P_FP8) return TN == 128 ? ((r >> 1) & 3) << 1 : ((r >> 2) & 1) << 1;
  else if constexpr (PREC == P_BF16) return TN == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2;
  else return ((r >> 2) & 1) << 3;
}

// One stage of an operand in registers: R rows (KC: R tile rows of 128 bytes of k; else
// R = columns, 128 / EB k-rows of R * EB bytes) spread over NT threads in 16-byte chunks.
// Past the group's range of k the stage is zero and costs no memory access (KC lanes there
// get an offset outside the resource, k-rows there lie outside it), so the pipeline below
// issues its loads without conditions and waits for exactly the stage that it stores.
template <int PREC, int R, int NT, bool KC>
struct Stage {
  static constexpr int EB = elem_bytes<PREC>();
  static constexpr int CPR = KC ? kStage / 16 : R * EB / 16;  // chunks per LDS row
  static constexpr int NR = R * (kStage / 16) / NT;           // chunks per thread
  static constexpr int RPP = NT / CPR;                        // LDS rows per pass
  static_assert(NT % CPR == 0 && (R * (kStage / 16)) % NT == 0, "whole chunks per thread");
  u32x4 r[NR];

  // src: first row / column of the tile at k = k0; left: k-values left in the range
  __device__ __forceinline__ void load(const uint8_t* src, uint32_t ldb, int left, int t) {
    const uint32_t row = (uint32_t)t / CPR, ch = (uint32_t)t % CPR;
    uint32_t vo = row * ldb + ch * 16;
    if (KC && (int)ch * (16 / EB) >= left) vo = 0x80000000u;
    // a resource per pass: its base moves in 64 bits, lane offsets stay below 2^31
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int rest = KC ? 0x7FFFFFFF : min(max(left - h * RPP, 0), RPP) * (int)ldb;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(src) + (int64_t)(h * RPP) * ldb, (short)0,
          __builtin_amdgcn_readfirstlane(rest), 0x00020000);
      r[h] = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, 0, 0);
    }
  }

  __device__ __forceinline__ void store(uint8_t* lds, int t) const {
    const int row = t / CPR, ch = t % CPR;
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int rr = row + h * RPP;
      const int s = KC ? swz_k(rr) : swz_n<PREC, R>(rr);
      *reinterpret_cast<u32x4*>(lds + rr * (CPR * 16) + ((ch ^ s) << 4)) = r[h];
    }
  }
};

template <int PREC>
struct FragOf {
  typedef bf16x8 T;
};
template <>
struct FragOf<P_FP8> {
  typedef long T;
};
template <>
struct FragOf<P_F32> {
  typedef f32x4 T;
};

// Matrix fragment of rows r0 + lane % 32 of a k-contiguous tile, k-values kk + 8 (lane / 32)
// ... (float32: kk + 4 (lane / 32) ...).
template <int PREC>
__device__ __forceinline__ typename FragOf<PREC>::T frag_k(const uint8_t* lds, int r0, int kk,
                                                           int lane) {
  constexpr int EB = elem_bytes<PREC>();
  const int r = r0 + (lane & 31);
  const int kb = (kk + (k_span<PREC>() / 2) * (lane >> 5)) * EB;
  return *reinterpret_cast<const typename FragOf<PREC>::T*>(
      lds + r * kStage + (((kb >> 4) ^ swz_k(r)) << 4) + (kb & 15));
}

// The same fragment of columns n0 + lane % 32 of an n-contiguous tile. A transposing read
// works on 16 lanes: e4m3 8 k-rows x 16 columns, lane i addressing row i / 2 and columns
// 8 (i % 2); bf16 4 k-rows x 16 columns, lane i addressing row i / 4 and columns 4 (i % 4);
// lane i receives column i.
template <int PREC, int TN>
__device__ __forceinline__ typename FragOf<PREC>::T frag_n(const uint8_t* lds, int n0, int kk,
                                                           int lane) {
  constexpr int RB = TN * elem_bytes<PREC>();
  const int hi = lane >> 5, c16 = 16 * ((lane >> 4) & 1), i = lane & 15;
  if constexpr (PREC == P_FP8) {
    const int r = 8 * hi + (i >> 1), cb = n0 + c16 + 8 * (i & 1);
    const int o = (kk + r) * RB + (((cb >> 4) ^ swz_n<PREC, TN>(r)) << 4) + (cb & 15);
    return __builtin_bit_cast(long, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                        (__attribute__((address_space(3))) i32x2*)(lds + o)));
  } else if constexpr (PREC == P_BF16) {
    struct {
      i16x4 h[2];
    } v;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 8 * hi + 4 * h + (i >> 2), cb = (n0 + c16 + 4 * (i & 3)) * 2;
      const int o = (kk + r) * RB + (((cb >> 4) ^ swz_n<PREC, TN>(r)) << 4) + (cb & 15);
      v.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) i16x4*)(lds + o));
    }
    return __builtin_bit_cast(bf16x8, v);
  } else {
    f32x4 v;
    const int cb = (n0 + (lane & 31)) * 4;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = 4 * hi + u;
      v[u] = *reinterpret_cast<const float*>(
          lds + (kk + r) * RB + (((cb >> 4) ^ swz_n<PREC, TN>(r)) << 4) + (cb & 15));
    }
    return v;
  }
}

// acc += (A B)^T of one multiply step: a lane holds column m = lane % 32 of the transposed
// 32x32 tile and rows n = 8 (j / 4) + 4 (lane / 32) + j % 4.
template <int PREC>
__device__ __forceinline__ void mma(f32x16& acc, typename FragOf<PREC>::T a,
                                    typename FragOf<PREC>::T b) {
  if constexpr (PREC == P_F32) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[u], a[u], acc, 0, 0, 0);
  } else if constexpr (PREC == P_FP8) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(b, a, acc, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, acc, 0, 0, 0);
  }
}

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
  const uint8_t* A = reinterpret_cast<const uint8_t*>(g.A) + (int64_t)c * g.sA * EB +
                     (int64_t)(bm * TM) * lda + (int64_t)kfirst * EB;
  const uint8_t* B = reinterpret_cast<const uint8_t*>(g.B) + (int64_t)c * g.sB * EB +
                     (B_K ? (int64_t)(bn * TN) * ldb + (int64_t)kfirst * EB
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

  Stage<PREC, TM, NT, true> pa, qa;
  Stage<PREC, TN, NT, B_K> pb, qb;
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

// Tile of a GEMM: the largest that still gives every CU a block (one resident block of
// 96 KB for two groups, two of 64 KB for one), since a tile's operand traffic per output
// falls with its edges. Measured, Xb W1 and H1 W2 of 16 chains together: e4m3
// 3072-1024-1024, n = 512, one group: 128 x 128 (512 blocks) 71 us against 82 us with
// 64 x 128; bf16 3072-512-512, n = 256, two groups: 64 x 128 (256 blocks) 47 us against
// 54 us with 64 x 64. Float32 is bound by the matrix cores, and at few tiles by the number
// of SIMDs that have one: 32 x 64 tiles at 4 chains take 52 us where one group per K half
// in launches of their own took 81 us.
template <int PREC, bool B_K, int EPI>
void dispatch(const Gemm& g, const Step& s, hipStream_t st, int splits) {
  const int64_t blocks = (int64_t)(g.M / 64) * (g.N / 128) * s.C;  // of 64 x 128
  if (splits == 1) {
    if (g.M % 128 == 0 && blocks >= 1024) launch<PREC, 128, 128, 2, 2, 1, B_K, EPI>(g, s, st);
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
