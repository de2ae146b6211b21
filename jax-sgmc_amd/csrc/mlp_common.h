// State, formats and helpers shared by the kernels of the MLP engine (mlp.hip, mlp_fwd.hip).
#pragma once
#include <math.h>

#include "sgmc_common.h"
#include "sgmc_device.h"

namespace sgmc {
namespace mlp {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// GEMM operand precision (template argument) and its element bytes.
enum Prec { P_BF16 = 0, P_FP8 = 1, P_F32 = 2 };
template <int PREC>
constexpr int elem_bytes() {
  return PREC == P_FP8 ? 1 : PREC == P_BF16 ? 2 : 4;
}

constexpr int GT = 256;
constexpr int BM = 64;
constexpr int BN = 128;
constexpr int NCLS = 10;
constexpr int NLEAF = 6;     // W1, W2, W3, b1, b2, b3
constexpr int kStrip = 32;   // rows per partial sum of the small leaves' gradients
constexpr int kXcds = 8;         // accelerator complex dies, each with its own L2
constexpr int kFinalBlocks = 64;
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// OCP fp8 e4m3 with a per-tensor scale: q = e4m3(clamp(v * scale, +-448)), v = q / scale.
__device__ __forceinline__ uint8_t f2q(float v) {
  v = fminf(fmaxf(v, -448.0f), 448.0f);
  return (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false) & 0xFFu);
}
__device__ __forceinline__ float q2f(uint8_t b) { return __builtin_amdgcn_cvt_f32_fp8((int)b, 0); }

// Four values packed: bf16 (as f2bf) and e4m3 (as f2q).
typedef uint32_t u32x2_4 __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ u32x2_4 pack_bf(f32x4 v) {
  return u32x2_4{(uint32_t)f2bf(v.x) | ((uint32_t)f2bf(v.y) << 16),
                 (uint32_t)f2bf(v.z) | ((uint32_t)f2bf(v.w) << 16)};
}
__device__ __forceinline__ uint32_t pack_q(f32x4 v) {
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = fminf(fmaxf(v[u], -448.0f), 448.0f);
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v.x, v.y, 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v.z, v.w, lo, true);
}

// fp8 tensors and their per-chain scale words: scales [0, 6), the scale the next weight
// shadows are written with [6, 8), amax bit patterns [8, 14).
enum Q8 { Q_X = 0, Q_H1 = 1, Q_DA2 = 2, Q_DA1 = 3, Q_W1 = 4, Q_W2 = 5 };
constexpr int kQWords = 16;
constexpr float kQTarget = 224.0f;  // scale = kQTarget / amax: half the e4m3 range as headroom

enum Epi { EPI_BIAS_RELU = 0, EPI_MASK = 1, EPI_UPDATE = 2, EPI_GRAD = 3 };

// Per-chain state and step parameters shared by the kernels.
struct Step {
  const float* X;          // dataset [N][ldx] float32
  const int32_t* labels;   // [N]
  int64_t N, ldx;
  int D_in, H1, H2, n, C;
  float* theta;            // [C][P]
  float* v;                // [C][P] or null (rms_prop)
  uint16_t* shadow;        // [C][P] bf16 (null for float32 GEMMs)
  int64_t P;
  int64_t off[NLEAF];      // leaf offsets
  int64_t size[NLEAF];     // leaf sizes
  uint32_t* key;           // [C][2]
  uint32_t* dkey;          // [C][2]
  uint32_t* lkey;          // [C][NLEAF][2] noise keys of this update, written by the gather
  uint32_t rmult, rmagic;  // randint_mult(N), randint_magic(N) of the index draw
  // activations: bf16; e4m3 except h2 (bf16) in fp8 mode; float32 in fp32 mode
  void* Xb;                // [C][n][D_in]
  int32_t* lab;            // [C][n]
  void* h1;                // [C][n][H1]
  void* h2;                // [C][n][H2]
  void* da2;               // [C][n][H2]
  void* da1;               // [C][n][H1]
  float* dL;               // [C][n][10]
  float* lik;              // [C][n]
  float* prior_part;       // [C][nparts]
  int nparts;
  float* U;                // [C]
  float* grad;             // [C][P] (gradient-only mode) or null
  float* samples;          // [C][n_slots][P] or null
  float* samples_U;        // [C][n_slots] or null
  int n_slots;
  const float* eps_table;
  const int32_t* save_slot;
  int32_t* iter;
  unsigned* counters;      // [C] arrival counters of the small kernel
  unsigned* done;
  int table_len;
  int rms;
  int update;              // 0: gradient only (autograd backward)
  float alpha, lmbd, temperature, noise_temperature;
  float prior_inv_var, prior_log_norm;
  int has_prior;
  // OBABO (update != 0, mode != MLP_SGLD)
  int mode;
  float* mom;              // [C][P] momentum
  float* ke_part;          // [C][nparts] kinetic-energy partials of one evaluation
  float* col_part;         // [C][n / kStrip][small leaves] row-strip gradient partials
  double* facc;            // [C] float64 likelihood of the full pass's chunks before this one
  double* fin_part;        // [C][kFinalBlocks] log-prior partials of the full pass
  double* ke;              // [C][2] accumulated kinetic energy at start / end
  float* U_half;           // [C] potential of the step's first evaluation
  const float* decay_table;  // [table_len] sqrt(exp(-friction eps))
  const float* noise_table;  // [table_len] sqrt((1 - exp(-friction eps)) T)
  // full-data forward pass (likelihoods of rows row0 .. row0 + n - 1 only)
  int full;
  int64_t row0;
  // fp8 GEMM operands (Xb, h1, da2, da1 and the W1 / W2 shadows in e4m3)
  int fp8;
  int fp32;                // float32 activations and GEMM operands (weights from theta)
  int split[3];            // split-K factors of G1, G2, G3
  float* q;                // [C][kQWords]
  uint8_t* shadow8;        // [C][P] (W1 and W2 leaves)
};

// Records max |v| of a wavefront for tensor t of chain c (every lane of the wavefront
// calls this). The atomic is skipped when the recorded maximum already covers the
// wavefront's: thousands of wavefronts updating one word otherwise serialize at the L2.
// A stale read is never above the true maximum, so no needed update is skipped.
__device__ __forceinline__ void q_note_amax(const Step& s, int c, int t, float a) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) a = fmaxf(a, __shfl_xor(a, m, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0 && a > 0.0f) {
    unsigned* slot = reinterpret_cast<unsigned*>(s.q + (int64_t)c * kQWords + 8 + t);
    const unsigned cur = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__float_as_uint(a) > cur) atomicMax(slot, __float_as_uint(a));
  }
}

// Block-wide version (every thread of the block calls it): one check and at most one
// atomic per block, for kernels whose wavefronts are too short to carry their own.
__device__ __forceinline__ void q_note_amax_block(const Step& s, int c, int t, float a,
                                                  float* red) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) a = fmaxf(a, __shfl_xor(a, m, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    float b = red[0];
    for (int i = 1; i < (int)(blockDim.x / kWave); ++i) b = fmaxf(b, red[i]);
    if (b > 0.0f) {
      unsigned* slot = reinterpret_cast<unsigned*>(s.q + (int64_t)c * kQWords + 8 + t);
      const unsigned cur = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__float_as_uint(b) > cur) atomicMax(slot, __float_as_uint(b));
    }
  }
}

enum MlpMode { MLP_SGLD = 0, MLP_OBABO_BA = 1, MLP_OBABO_BO = 2 };

__device__ __forceinline__ int cur_iter(const Step& s) {
  return max(0, min(s.iter[0], s.table_len - 1));
}


// ------------------------------------------------------------------ GEMM ------
// Operands are bf16, e4m3 (P_FP8) with per-tensor scales, or float32 (P_F32): element
// pointers are byte addresses of 2-, 1- or 4-byte elements, strides are in elements.
struct Gemm {
  const void* A;
  int64_t lda, sA;   // sA: chain stride in elements
  const void* B;
  int64_t ldb, sB;
  int M, N, K;
  void* out;         // EPI_BIAS_RELU / EPI_MASK
  int64_t ldo, sO;
  const float* bias; // chain-strided by sBias
  int64_t sBias;
  const void* mask;  // EPI_MASK: ReLU activations (same format as the operands)
  int64_t ldm, sM;
  int leaf;          // EPI_UPDATE / EPI_GRAD: parameter leaf of the [M][N] weight
  int part0;         // first prior-partial slot of this GEMM
  int ta, tb;        // P_FP8: scale slots of A and B
  int tout;          // P_FP8: scale slot of an e4m3 output, or -1 for a bf16 output
};

// GEMM call sites of one evaluation (the tune[] slots): G1 = Xb W1, G2 = H1 W2,
// G3 = dA2 W2^T, G4 = H1^T dA2 (gW2), G5 = Xb^T dA1 (gW1).
enum GemmSlot { SLOT_G1 = 0, SLOT_G2, SLOT_G3, SLOT_G4, SLOT_G5, kSlots };

// ReLU mask of an activation element (bf16, e4m3 or float32): positive and nonzero.
template <int PREC>
__device__ __forceinline__ bool mask_on(const void* m, int64_t i) {
  if constexpr (PREC == P_F32) {
    const uint32_t u = __float_as_uint(reinterpret_cast<const float*>(m)[i]);
    return u != 0 && !(u & 0x80000000u);
  } else if constexpr (PREC == P_FP8) {
    const uint8_t b = reinterpret_cast<const uint8_t*>(m)[i];
    return b != 0 && !(b & 0x80u);
  } else {
    const uint16_t h = reinterpret_cast<const uint16_t*>(m)[i];
    return h != 0 && !(h & 0x8000u);
  }
}

// Writes an activation: float32 (f32), e4m3 at scale qs (q8), or bf16.
__device__ __forceinline__ void put_act(void* out, int64_t i, float v, bool q8, float qs,
                                        bool f32) {
  if (f32) reinterpret_cast<float*>(out)[i] = v;
  else if (q8) reinterpret_cast<uint8_t*>(out)[i] = f2q(v * qs);
  else reinterpret_cast<uint16_t*>(out)[i] = f2bf(v);
}

// The activation GEMMs G1-G3 (bias and ReLU, or a ReLU mask where g.mask is set), K split
// over `splits` groups of wavefronts (1 to 4).
void launch_act_gemm(const Gemm& g, const Step& s, hipStream_t st, int splits);

// The parameter GEMMs gW2 (g4) and gW1 (g5) with their update (s.update) or gradient.
void launch_param_gemms(const Gemm& g4, const Gemm& g5, const Step& s, hipStream_t st);

// Bytes per element of an activation tensor written with (q8, f32).
__device__ __forceinline__ int act_bytes(bool q8, bool f32) { return f32 ? 4 : q8 ? 1 : 2; }

}  // namespace mlp
}  // namespace sgmc
