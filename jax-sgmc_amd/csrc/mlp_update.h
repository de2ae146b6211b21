// The parameter update of the MLP engine (SGLD, rms_prop, OBABO halves), shared by the
// parameter GEMMs (mlp_param.hip) and the small leaves' kernel (mlp.hip).
#pragma once
#include "mlp_common.h"

namespace sgmc {
namespace mlp {

// Parameter update of one leaf of chain c, applied to values so that a thread can
// issue the loads of all its parameters before the arithmetic. The leaf's arrays are
// addressed from uniform base pointers with 32-bit offsets (a leaf holds < 2^32
// entries). Update rules (prior gradient and temperature folded into g = (gsum + w /
// s^2) / T, written with fused multiply-adds: within an ulp or two of the reference's
// separate roundings, far inside the bf16 / e4m3 GEMM error):
//   SGLD (integrator.py:882-912): w += (-eps) g + sqrt(2 T eps) xi; with rms_prop
//     (adaption.py:254-291): v = alpha v + (1 - alpha) g^2, G = 1 / (lmbd + sqrt(v)),
//     w += G (-eps) g + sqrt(G) sqrt(2 T eps) xi (hardware reciprocal and square roots);
//   OBABO with the identity mass (integrator.py:181-273), in two halves:
//     BA: p1 = sqrt(pi) p + sqrt((1 - pi) T) xi(s1); KE_start += p1^2 / 2;
//         p2 = (-eps/2) g + p1; w += eps p2
//     BO: p3 = (-eps/2) g(w') + p2; KE_end += p3^2 / 2; p = sqrt(pi) p3 + ... xi(s2).
struct Upd {
  float* th;          // theta of the leaf
  float* aux;         // rms_prop v or OBABO momentum of the leaf, or null (plain SGLD)
  uint16_t* sh;       // bf16 shadow of the leaf, or null
  uint8_t* sh8;       // e4m3 shadow (W1, W2 in fp8 mode), or null
  float q8;           // scale the e4m3 shadow is written with
  int mode, rms, has_prior;
  float inv_var, log_norm, inv_T, eps, noise_scale, decay, noise, half, alpha, one_m_alpha,
      lmbd;
};

// Per-kernel step coefficients of the current iteration.
struct Coef {
  float eps, noise_scale, decay, noise;
};

__device__ __forceinline__ Coef coef_of(const Step& s) {
  const int it = cur_iter(s);
  Coef k;
  k.eps = s.eps_table[it];
  k.noise_scale = sqrtf((2.0f * s.noise_temperature) * k.eps);
  k.decay = s.decay_table ? s.decay_table[it] : 0.0f;
  k.noise = s.noise_table ? s.noise_table[it] : 0.0f;
  return k;
}

__device__ __forceinline__ Upd make_upd(const Step& s, int c, int leaf, int64_t base,
                                        const Coef& k) {
  Upd u;
  u.th = s.theta + base;
  u.aux = s.mode == MLP_SGLD ? (s.rms ? s.v + base : nullptr) : s.mom + base;
  u.sh = nullptr;
  u.sh8 = nullptr;
  u.q8 = 1.0f;
  if (s.fp8 && leaf < 2) {
    u.sh8 = s.shadow8 + base;
    u.q8 = s.q[(int64_t)c * kQWords + 6 + leaf];
  } else if (!s.fp32) {
    u.sh = s.shadow + base;
  }
  u.mode = s.mode;
  u.rms = s.rms;
  u.has_prior = s.has_prior;
  u.inv_var = s.prior_inv_var;
  u.log_norm = s.prior_log_norm;
  u.inv_T = 1.0f / s.temperature;
  u.eps = k.eps;
  u.noise_scale = k.noise_scale;
  u.decay = k.decay;
  u.noise = k.noise;
  u.half = 0.5f * k.eps;
  u.alpha = s.alpha;
  u.one_m_alpha = 1.0f - s.alpha;
  u.lmbd = s.lmbd;
  return u;
}

// UM: the update rule compiled in -- UM_RMS: SGLD with rms_prop (state v in aux);
// UM_OBA / UM_OBO: the O B A and B O halves of an OBABO step (momentum in aux); or
// UM_ANY: the rule of u.mode / u.rms at run time.
constexpr int UM_ANY = 0;
constexpr int UM_RMS = 1;
constexpr int UM_OBA = 2;
constexpr int UM_OBO = 3;

// the rule's mode
template <int UM>
__device__ __forceinline__ int um_mode(const Upd& u) {
  return UM == UM_RMS ? MLP_SGLD : UM == UM_OBA ? MLP_OBABO_BA : UM == UM_OBO ? MLP_OBABO_BO
                                                                               : u.mode;
}

__device__ __forceinline__ void upd_load(const Upd& u, uint32_t i, float& w, float& aux) {
  w = u.th[i];
  aux = u.aux ? u.aux[i] : 0.0f;
}

template <int UM = UM_ANY>
__device__ __forceinline__ void upd_step(const Upd& u, float& w, float& aux, float gsum,
                                         float xi, float& lp, float& ke) {
  float g = gsum;
  if (u.has_prior) {
    g = __builtin_fmaf(w, u.inv_var, g);
    lp = __builtin_fmaf(__builtin_fmaf(w * w, u.inv_var, u.log_norm), -0.5f, lp);
  }
  g = g * u.inv_T;
  const int mode = um_mode<UM>(u);
  if (mode == MLP_SGLD) {
    const float sg = (-u.eps) * g;
    const float sn = u.noise_scale * xi;
    if (UM == UM_RMS || u.rms) {
      const float vn = __builtin_fmaf(u.alpha, aux, u.one_m_alpha * (g * g));
      aux = vn;
      // G = 1 / (lambda + sqrt(v)) and sqrt(G) from one reciprocal square root
      const float rG = __builtin_amdgcn_rsqf(u.lmbd + __builtin_amdgcn_sqrtf(vn));
      w = w + __builtin_fmaf(rG, sn, (rG * rG) * sg);
    } else {
      w = w + (sg + sn);
    }
  } else if (mode == MLP_OBABO_BA) {
    const float p1 = __builtin_fmaf(u.decay, aux, u.noise * xi);
    ke = __builtin_fmaf(p1, p1, ke);
    const float p2 = __builtin_fmaf(-u.half, g, p1);
    aux = p2;
    w = __builtin_fmaf(u.eps, p2, w);
  } else {
    const float p3 = __builtin_fmaf(-u.half, g, aux);
    ke = __builtin_fmaf(p3, p3, ke);
    aux = __builtin_fmaf(u.decay, p3, u.noise * xi);
  }
}

__device__ __forceinline__ void upd_store(const Upd& u, uint32_t i, float w, float aux,
                                          float& wmax) {
  if (u.mode != MLP_OBABO_BO) {
    u.th[i] = w;
    if (u.sh8) {
      u.sh8[i] = f2q(w * u.q8);
      wmax = fmaxf(wmax, fabsf(w));
    } else if (u.sh) {
      u.sh[i] = f2bf(w);
    }
  }
  if (u.aux) u.aux[i] = aux;
}

// Key of leaf `leaf` of the noise tree of this update: random_tree(sub) with
// (key, sub) = split(key) for SGLD; s1 / s2 of (key, s1, s2) = split(key, 3) for the
// two momentum refreshes of an OBABO step.
__device__ __forceinline__ Key derive_leaf_key(const Step& s, int chain, int leaf) {
  const Key k = load_key(s.key + 2 * chain);
  Key a, b, c;
  if (s.mode == MLP_SGLD) {
    split2(k, a, b);
    return split_key(b, NLEAF, (uint32_t)leaf);
  }
  split3(k, a, b, c);
  return split_key(s.mode == MLP_OBABO_BA ? b : c, NLEAF, (uint32_t)leaf);
}

// The same key as stored by the step's gather kernel (the chain key does not change
// until the step's last kernel), so the update epilogues load two words instead of
// running four to seven Threefry blocks per wave.
__device__ __forceinline__ Key leaf_key(const Step& s, int chain, int leaf) {
  return load_key(s.lkey + 2 * (chain * NLEAF + leaf));
}

}  // namespace mlp
}  // namespace sgmc
