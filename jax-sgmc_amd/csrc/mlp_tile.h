// Operand stages, fragments and multiply step of the MLP engine's GEMMs (mlp_fwd.hip,
// mlp_param.hip).
#pragma once
#include "mlp_common.h"

namespace sgmc {
namespace mlp {

constexpr int kStage = 128;  // bytes of k per row and stage

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

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

  // First row of this wavefront in a pass over a k-contiguous tile. Its resources begin there,
  // with a base of 64 bits, so that lane offsets span eight rows and stay below 2^31 at every
  // accepted width (over all rows of a pass they went past it at inputs of 17 M float32
  // columns). A pass over an n-contiguous tile spans 16 NT / R <= 64 bytes per column of the
  // operand, below 2^31 for fewer than 2^25 columns, and begins at row 0.
  static __device__ __forceinline__ int first(int t) {
    return KC ? __builtin_amdgcn_readfirstlane(t / kWave) * (kWave / CPR) : 0;
  }

  // src: row first(t) (n-contiguous: first column) of the tile at k = k0; left: k-values left
  // in the range; gap: bytes between the two halves of a row's columns that lie apart
  // (n-contiguous tiles)
  __device__ __forceinline__ void load(const uint8_t* src, uint32_t ldb, int left, int t,
                                       uint32_t gap = 0) {
    const uint32_t row = (uint32_t)(KC ? t % kWave : t) / CPR, ch = (uint32_t)t % CPR;
    uint32_t vo = row * ldb + ch * 16 + (ch >= CPR / 2 ? gap : 0);
    if (KC && (int)ch * (16 / EB) >= left) vo = 0x80000000u;
    // a resource per pass: its base moves in 64 bits
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
      u32x4 v = r[h];
      if (KC && PREC == P_FP8 && (rr & 16)) v = u32x4{v.z, v.w, v.x, v.y};  // see frag_k
      *reinterpret_cast<u32x4*>(lds + rr * (CPR * 16) + ((ch ^ s) << 4)) = v;
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
// ... (float32: kk + 4 (lane / 32) ...). e4m3 takes half a chunk per lane: rows with bit 4 set
// hold a chunk's halves swapped, so the 32 rows that one half-wavefront reads use both (in one
// half of the chunks they met two by two on the banks, 20% of the LDS cycles).
template <int PREC>
__device__ __forceinline__ typename FragOf<PREC>::T frag_k(const uint8_t* lds, int r0, int kk,
                                                           int lane) {
  constexpr int EB = elem_bytes<PREC>();
  const int r = r0 + (lane & 31);
  const int kb = (kk + (k_span<PREC>() / 2) * (lane >> 5)) * EB;
  const int half = PREC == P_FP8 ? (kb & 15) ^ ((r & 16) >> 1) : kb & 15;
  return *reinterpret_cast<const typename FragOf<PREC>::T*>(
      lds + r * kStage + (((kb >> 4) ^ swz_k(r)) << 4) + half);
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

}  // namespace mlp
}  // namespace sgmc
