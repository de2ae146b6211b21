// The parameter GEMMs of the MLP engine, gW1 = Xb^T dA1 and gW2 = H1^T dA2, with the
// parameter update (or the gradient's store) in the epilogue, in one launch.
//
// What bounds them: the update's state. A pSGLD step of 16 chains of 3072-512-512 streams
// 29 M parameters' theta, v and bf16 copy, 530 MB (103 us at the 5.2 TB/s of a large copy),
// and each parameter's share of a Threefry block, its normal and its update is about 80
// vector instructions, 75 us for the chip; the matrix work is 6 us. So the product is only
// a short prologue: both operands go to LDS as they lie (k rows) and are read with the
// transposing LDS loads, the products then move through LDS so that a thread owns four
// consecutive columns of a row and of the row half the leaf further (the two words of one
// Threefry block, integrator.py:119-135), its state moves in 16-byte accesses that cover
// whole lines, and the first of them are in flight before the product is begun.
// Against a lane per parameter pair, 4-byte accesses and operands transposed in registers:
// that step's update 163 -> 121 us (611 MB beyond the L2 with the operands, 5.0 TB/s); 16
// chains of 3072-1024-1024 in e4m3, n = 512: OBA half 378 -> 279 us, BO half 252 -> 204 us,
// gradient 210 -> 161 us; float32 gradient of 4 chains of 3072-512-512 55 -> 47 us.
#include "mlp_colsum.h"
#include "mlp_tile.h"
#include "mlp_update.h"

namespace sgmc {
namespace mlp {
namespace {

// Three waves per SIMD: at four (128 registers) the OBABO update of e4m3 operands spills
// (16 chains of 3072-1024-1024: 295 us against 279).
constexpr int kWavesPerSimd = 3;
constexpr int kRawBufferFlags = 0x00020000;  // word 3 of a raw buffer resource (CDNA)

// 2^32 - 16 bytes from p: the 32 rows of a band span less at the widest layer (a leaf has fewer
// than 2^32 entries and at least 128 rows or columns: rows of up to 2^25 floats).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, bool on = true) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, on ? (int)0xFFFFFFF0u : 0,
                                           kRawBufferFlags);
}
// State is stored with the non-temporal hint, which leaves the last-level cache to what the
// next evaluation reads (the GEMM copies and X): pSGLD, 16 chains of 3072-512-512, Xb W1
// 39 -> 35 us and the gather 25 -> 24 us at the same update time. Loads with the hint lose
// more here (121 -> 143 us) than they give there.
constexpr int kNonTemporal = 2;
__device__ __forceinline__ f32x4 ld4(__amdgpu_buffer_rsrc_t r, uint32_t bytes) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, bytes, 0, 0));
}
__device__ __forceinline__ void st4(f32x4 v, __amdgpu_buffer_rsrc_t r, uint32_t bytes) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, bytes, 0,
                                         kNonTemporal);
}

typedef uint32_t u32_2 __attribute__((aligned(2)));  // e4m3 copies of odd chains

constexpr int BW = 32;  // 64 x 64 tiles: 134 us for 124 (pSGLD), 316 for 295 (e4m3 OBA)

// Block `lin` of a GEMM: 2 BW rows of the leaf (BW and, half the leaf further, BW more) by
// TN = 4096 / BW columns, chain c. Four wavefronts of 64 x 32 each.
template <int PREC, int EPI, int UM>
__device__ __forceinline__ void param_tile(const Gemm& g, const Step& s, uint32_t lin,
                                           uint32_t gx, uint32_t gy, uint8_t* lds, float* red) {
  constexpr bool F8 = PREC == P_FP8;
  constexpr int EB = elem_bytes<PREC>();
  constexpr int W = 2 * BW, TN = 4096 / BW, WM = W / 64;
  constexpr int KE = kStage / EB;
  // XCD x takes the contiguous range [x T / 8, (x + 1) T / 8) of tiles, n fastest, then m,
  // then chain: the blocks that share operand rows read them through one L2 and a leaf's
  // rows are written whole. Against m fastest over all XCDs (16 chains): the e4m3 updates
  // of 3072-1024-1024 326 -> 279 us (OBA) and 210 -> 204 us (BO), pSGLD 3072-512-512 125 ->
  // 124 us.
  const uint32_t T = gx * gy * (uint32_t)s.C;
  if (T % kXcds == 0) lin = (lin % kXcds) * (T / kXcds) + lin / kXcds;
  const int bn = (int)(lin % gy), bm = (int)((lin / gy) % gx), c = (int)(lin / (gx * gy));
  const int t = (int)threadIdx.x, lane = t & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const int m0 = (w % WM) * 64, n0 = (w / WM) * 32;
  const int half = g.M / 2;

  // this thread's parameters: rows r0 + kRows i (and half further) of the tile, 4 columns
  constexpr int kQuads = TN / 4, kRows = GT / kQuads, kIts = BW / kRows;
  const int qd = t % kQuads, r0 = t / kQuads;
  const int64_t leaf0 = (int64_t)c * s.P + s.off[g.leaf];
  const int64_t tile0 = (int64_t)(bm * BW) * g.N + bn * TN, tile1 = tile0 + (int64_t)half * g.N;
  const uint32_t e0 = (uint32_t)r0 * (uint32_t)g.N + 4 * qd;  // of the tile
  auto elem = [&](int i) __attribute__((always_inline)) -> uint32_t {
    return e0 + (uint32_t)(i * kRows) * (uint32_t)g.N;
  };
  const Coef k = coef_of(s);
  const Upd up = make_upd(s, c, g.leaf, leaf0, k);
  const bool has_aux = EPI == EPI_UPDATE && (UM != UM_ANY || up.aux);
  const __amdgpu_buffer_rsrc_t th0 = rsrc(up.th + tile0), th1 = rsrc(up.th + tile1);
  const __amdgpu_buffer_rsrc_t au0 = rsrc(up.aux + tile0, has_aux),
                               au1 = rsrc(up.aux + tile1, has_aux);
  f32x4 w0, w1, a0{}, a1{};
  auto fetch = [&](int i) __attribute__((always_inline)) {
    w0 = ld4(th0, 4 * elem(i));
    w1 = ld4(th1, 4 * elem(i));
    if constexpr (EPI == EPI_UPDATE) {
      a0 = ld4(au0, 4 * elem(i));
      a1 = ld4(au1, 4 * elem(i));
    }
  };
  fetch(0);
  __builtin_amdgcn_sched_barrier(0);

  f32x16 acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  const uint32_t lda = (uint32_t)(g.lda * EB), ldb = (uint32_t)(g.ldb * EB);
  const uint8_t* A = reinterpret_cast<const uint8_t*>(g.A) + (int64_t)c * g.sA * EB +
                     (int64_t)(bm * BW) * EB;
  const uint8_t* B = reinterpret_cast<const uint8_t*>(g.B) + (int64_t)c * g.sB * EB +
                     (int64_t)(bn * TN) * EB;
  const uint32_t gap = (uint32_t)((half - BW) * EB);
  Stage<PREC, W, GT, false> pa;
  Stage<PREC, TN, GT, false> pb;
  uint8_t* const Bs = lds + W * kStage;
  auto load = [&](int k0) __attribute__((always_inline)) {
    pa.load(A + (int64_t)k0 * lda, lda, g.K - k0, t, gap);
    pb.load(B + (int64_t)k0 * ldb, ldb, g.K - k0, t);
    __builtin_amdgcn_sched_barrier(0);
  };
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += KE) {
    pa.store(lds, t);
    pb.store(Bs, t);
    load(k0 + KE);
    lds_sync();
#pragma unroll
    for (int kk = 0; kk < KE; kk += k_span<PREC>()) {
      const auto b = frag_n<PREC, TN>(Bs, n0, kk, lane);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        mma<PREC>(acc[i], frag_n<PREC, W>(lds, m0 + 32 * i, kk, lane), b);
    }
    lds_sync();
  }

  // products to LDS, four consecutive columns per write, swizzled by the row
  float* const prod = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + 32 * i + (lane & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int q = (n0 + 8 * e) / 4 + (lane >> 5);
      *reinterpret_cast<f32x4*>(prod + m * TN + 4 * (q ^ (m & (kQuads - 1)))) =
          f32x4{acc[i][4 * e], acc[i][4 * e + 1], acc[i][4 * e + 2], acc[i][4 * e + 3]};
    }
  }
  lds_sync();

  const float* qc = F8 ? s.q + (int64_t)c * kQWords : nullptr;
  const float ab = F8 ? 1.0f / (qc[g.ta] * qc[g.tb]) : 1.0f;  // undoes the operand scales
  const uint32_t S = (uint32_t)((int64_t)g.M * g.N);
  float lp = 0.0f, ke = 0.0f, wmax = 0.0f;
  Key lk{};
  if constexpr (EPI == EPI_UPDATE) lk = leaf_key(s, c, g.leaf);
#pragma unroll
  for (int i = 0; i < kIts; ++i) {
    const uint32_t el = elem(i);
    const int m = r0 + i * kRows;
    const int po = 4 * (qd ^ (m & (kQuads - 1)));  // (BW is a multiple of kQuads: same for both)
    static_assert(BW % kQuads == 0, "one swizzle for both bands");
    const f32x4 p0 = *reinterpret_cast<const f32x4*>(prod + m * TN + po);
    const f32x4 p1 = *reinterpret_cast<const f32x4*>(prod + (BW + m) * TN + po);
    f32x4 x0 = w0, x1 = w1, y0 = a0, y1 = a1;
    if (i + 1 < kIts) fetch(i + 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EPI == EPI_UPDATE) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint32_t b0, b1;
        bits_pair(lk, S, (uint32_t)tile0 + el + u, b0, b1);
        float wa = x0[u], aa = y0[u], wb = x1[u], ab_ = y1[u];
        upd_step<UM>(up, wa, aa, ab * p0[u], bits_to_normal_fast(b0), lp, ke);
        upd_step<UM>(up, wb, ab_, ab * p1[u], bits_to_normal_fast(b1), lp, ke);
        x0[u] = wa;
        y0[u] = aa;
        x1[u] = wb;
        y1[u] = ab_;
      }
      if (um_mode<UM>(up) != MLP_OBABO_BO) {
        st4(x0, th0, 4 * el);
        st4(x1, th1, 4 * el);
        if constexpr (PREC == P_FP8) {
          *reinterpret_cast<u32_2*>(up.sh8 + tile0 + el) = pack_q(x0 * up.q8);
          *reinterpret_cast<u32_2*>(up.sh8 + tile1 + el) = pack_q(x1 * up.q8);
#pragma unroll
          for (int u = 0; u < 4; ++u) wmax = fmaxf(wmax, fmaxf(fabsf(x0[u]), fabsf(x1[u])));
        } else if constexpr (PREC == P_BF16) {
          *reinterpret_cast<u32x2_4*>(up.sh + tile0 + el) = pack_bf(x0);
          *reinterpret_cast<u32x2_4*>(up.sh + tile1 + el) = pack_bf(x1);
        }
      }
      if (has_aux) {
        st4(y0, au0, 4 * el);
        st4(y1, au1, 4 * el);
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 p = h ? p1 : p0, x = h ? x1 : x0;
        f32x4 o;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float gg = ab * p[u];
          if (s.has_prior) {
            gg = gg + x[u] * s.prior_inv_var;
            lp += (s.prior_log_norm + (x[u] * x[u]) * s.prior_inv_var) / -2.0f;
          }
          o[u] = gg / s.temperature;
        }
        *reinterpret_cast<f32x4u*>(s.grad + leaf0 + (h ? tile1 : tile0) + el) = o;
      }
    }
  }
  if constexpr (EPI == EPI_UPDATE && F8)
    if (UM != UM_OBO) q_note_amax_block(s, c, Q_W1 + g.leaf, wmax, red);
  const int64_t slot = (int64_t)c * s.nparts + g.part0 + bm * (int)gy + bn;
  const float tot = block_sum<GT>(lp, red);
  if (threadIdx.x == 0) s.prior_part[slot] = tot;
  if (EPI == EPI_UPDATE && UM != UM_RMS && s.mode != MLP_SGLD) {
    const float kt = block_sum<GT>(ke, red);
    if (threadIdx.x == 0) s.ke_part[slot] = kt;
  }
}

// A 1-D grid of both GEMMs. Every other update (odd iterations; the second half of an OBABO
// step) runs through it backwards, so that it begins with the state which the one before
// wrote last and the last-level cache still holds (pSGLD 3072-512-512, 16 chains: iteration
// 244 -> 237 us of kernels). The first blocks take gW1's tiles (ga) and the rest gW2's (gb), so
// gW2's fill the last round of gW1's. Ahead of both come the ncol blocks of the small leaves'
// column sums (colx per strip), which need the same activations and none of the parameters:
// latency-bound on their own (20 us in e4m3, 8 in bf16, 6 in float32), here they run beside the
// update (16 chains of 3072-512-512 bf16 121 + 8 -> 125 us, 4 chains in float32 47 + 6 -> 47).
template <int PREC, int EPI, int UM>
__global__ void __launch_bounds__(GT, kWavesPerSimd)
    param_kernel(Gemm ga, Gemm gb, Step s, uint32_t gxa, uint32_t gya, uint32_t gxb, uint32_t gyb,
                 uint32_t ncol, uint32_t colx) {
  constexpr int kProd = 2 * 4096 * 4, kStages = (2 * BW + 4096 / BW) * kStage;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kProd > kStages ? kProd : kStages];
  __shared__ float red[GT / kWave];
  if (blockIdx.x < ncol) {
    const uint32_t strips = (uint32_t)(s.n / kStrip), b = blockIdx.x;
    if (b < colx * strips * (uint32_t)s.C)
      colsum_block<PREC>(s, (int)(b % colx), (int)(b / colx % strips), (int)(b / (colx * strips)),
                         reinterpret_cast<float*>(lds));
    return;
  }
  const uint32_t na = gxa * gya * (uint32_t)s.C;
  const bool rev = s.mode == MLP_SGLD ? (cur_iter(s) & 1) != 0 : s.mode == MLP_OBABO_BO;
  const uint32_t lin = rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x - ncol;
  if (lin < na)
    param_tile<PREC, EPI, UM>(ga, s, lin, gxa, gya, lds, red);
  else
    param_tile<PREC, EPI, UM>(gb, s, lin - na, gxb, gyb, lds, red);
}

template <int PREC, int EPI, int UM>
void launch(const Gemm& ga, const Gemm& gb, const Step& s, hipStream_t st) {
  constexpr int W = 2 * BW, TN = 4096 / BW;
  const uint32_t gxa = (uint32_t)(ga.M / W), gya = (uint32_t)(ga.N / TN);
  const uint32_t gxb = (uint32_t)(gb.M / W), gyb = (uint32_t)(gb.N / TN);
  // the column sums' blocks first, padded to whole rounds over the XCDs
  const uint32_t colx = (uint32_t)colsum_blocks(s);
  const uint32_t ncol = (colx * (uint32_t)(s.n / kStrip) * (uint32_t)s.C + kXcds - 1) / kXcds * kXcds;
  hipLaunchKernelGGL((param_kernel<PREC, EPI, UM>),
                     dim3(ncol + (gxa * gya + gxb * gyb) * (uint32_t)s.C), dim3(GT), 0, st, ga, gb,
                     s, gxa, gya, gxb, gyb, ncol, colx);
}

// the update rule compiled in: rms_prop SGLD and the two OBABO halves; plain SGLD at run time
template <int PREC>
void by_rule(const Gemm& ga, const Gemm& gb, const Step& s, hipStream_t st) {
  if (!s.update) launch<PREC, EPI_GRAD, UM_ANY>(ga, gb, s, st);
  else if (s.mode == MLP_OBABO_BA) launch<PREC, EPI_UPDATE, UM_OBA>(ga, gb, s, st);
  else if (s.mode == MLP_OBABO_BO) launch<PREC, EPI_UPDATE, UM_OBO>(ga, gb, s, st);
  else if (s.rms) launch<PREC, EPI_UPDATE, UM_RMS>(ga, gb, s, st);
  else launch<PREC, EPI_UPDATE, UM_ANY>(ga, gb, s, st);
}

}  // namespace

void launch_param_gemms(const Gemm& g4, const Gemm& g5, const Step& s, hipStream_t st) {
  if (s.fp32) by_rule<P_F32>(g5, g4, s, st);
  else if (s.fp8) by_rule<P_FP8>(g5, g4, s, st);
  else by_rule<P_BF16>(g5, g4, s, st);
}

}  // namespace mlp
}  // namespace sgmc
