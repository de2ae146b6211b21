// The fused multi-chain GLM step and the loop over many iterations: kernels and their
// launch templates. Each sampler mode is compiled in a translation unit of its own
// (glm_fused_*.hip, glm_loop_*.hip instantiate the templates below).
#pragma once
#include "glm_rows.h"

namespace sgmc {


// ------------------------------------------------------------ fused path ----

struct FusedArgs {
  const sgmc_glm_chain* chains;
  const int32_t* block_chain;   // grid block -> chain, or NULL with blocks_per_chain
  int blocks_per_chain;         // uniform table: chain = block / blocks_per_chain
  const float* eps_table;
  const int32_t* save_slot;
  int32_t* iter;
  unsigned* done;
  const float* inv_mass;   // shared diagonal mass (nullable = ones)
  const float* sqrt_mass;
  int table_len;
  int nchains;
  int advance;             // the launch's last chain advances the iteration counter;
                           // < 0: no counter bookkeeping (the loop kernel does it)
  int iter_offset;         // iteration of this evaluation = *iter + iter_offset
  int step;                // leapfrog step within the iteration (SGHMC)
  int steps;
  float friction;
  float four_friction;     // float32(4 friction) (AMAGOLD noise scale)
  float alpha, lmbd;       // rms_prop
  Lik L;
  Prior pr;
  float pot_temperature;
};

// LDS of one fused block.
template <int MODE>
struct FusedLds {
  __attribute__((aligned(16))) float cols[kWaves * kMaxD];  // the wavefronts' column sums
  float small[4 * kWaves];                                   // reduction slots
  float lik[kLdsRows];
  float p[MODE == SGMC_MODE_SGHMC ? kMaxD : 1];              // resampled momentum
  int flag;
};

// Sums over the block of wave sums that every wavefront has put in slot[0 .. kWaves) before
// a barrier.
__device__ __forceinline__ float slot_sum(const float* slot) {
  float t = 0.0f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) t += slot[i];
  return t;
}
__device__ __forceinline__ void put_slot(float* slot, float v) {
  v = wave_sum(v);
  if ((threadIdx.x & (kWave - 1)) == 0) slot[threadIdx.x / kWave] = v;
}

// One evaluation of chain ch by its block bchain: draw, gather, likelihood, reduction, and
// in the chain's last block to arrive the update. MODE: the table's SGMC_MODE_*, fixed at
// compile time (the other modes' branches are folded away).
//
// A launch of small chains is a chain of latencies: descriptor, keys, index draw, rows,
// reduction, records, arrival, update. Everything that does not depend on the row sums is
// therefore done while something else is awaited: the key splits run as one Threefry block
// on two lanes each (split2_uniform), the step's noise, the resampled momentum and the
// evaluation point are formed behind the first rows' loads, the update's state is loaded
// with the arrival (every block loads it, 2 to 4 D floats; only the last uses it), the
// iteration counter is advanced beside the update, and the reductions share barriers.
// Per launch, from HIP graphs: 16 rms_prop chains (D = 100, n = 1000, 16 blocks each) 17.7 ->
// 15.7 us, 64 SGHMC chains (D = 12, n = 300) 13.1 -> 9.6, 4 OBABO chains (D = 300, n = 512,
// 16 blocks) 14.3 -> 11.3, one SGLD chain of 64 blocks (D = 300, n = 4096) 19.5 -> 14.8, 64
// SGHMC chains (D = 512, n = 4096, 4 blocks) 95.7 -> 93. What is left of a small chain's 9 us
// is the launch itself (2.5 us) and five dependent memory round trips.
template <int LPR, int CPL, int MODE>
__device__ __forceinline__ void fused_body(const FusedArgs& a, const sgmc_glm_chain& ch,
                                           int bchain, FusedLds<MODE>& lds) {
  constexpr bool hmc = MODE == SGMC_MODE_SGHMC;
  constexpr bool amg = MODE == SGMC_MODE_AMAGOLD;
  constexpr bool ob_mh = MODE == SGMC_MODE_SGGMC;
  constexpr bool ob = MODE == SGMC_MODE_OBABO || ob_mh;
  constexpr bool rms = MODE == SGMC_MODE_SGLD_RMS;
  constexpr bool has_mom = hmc || amg || ob;
  constexpr bool shift = hmc || amg;  // evaluation point theta + scale M^-1 p
  // noise pairs (j, j + m) of one thread
  constexpr int NP = 4 * LPR * CPL > 2 * kNT ? 2 : 1;
  const Key key0 = load_key(ch.key);
  const Key dkey0 = load_key(ch.dkey);
  const int it = max(0, min(a.iter[0] + a.iter_offset, a.table_len - 1));
  const float eps = a.eps_table[it];
  const int D = ch.D;
  const int D4 = (D + 3) >> 2;
  gfloat* g_theta = to_global(ch.theta);
  gfloat* g_mom = to_global(ch.mom);
  gfloat* g_v = to_global(ch.v);
  gfloat* g_partial = to_global(ch.partial);
  gfloat* g_lik = to_global(ch.lik);
  gfloat* g_samples = to_global(ch.samples);
  gcfloat* g_inv_mass = to_global(a.inv_mass);
  gcfloat* g_sqrt_mass = to_global(a.sqrt_mass);
  const bool resample = hmc && a.step == 0;
  // OBABO: two launches per leapfrog step, the even one O B A, the odd one B O.
  const int sub = a.step & 1;
  const int launches = ob ? 2 * a.steps : a.steps;
  // Position step before this evaluation: eps, or eps/2 at the first step of an
  // AMAGOLD iteration (integrator.py:521-523, 401-408).
  const float half = 0.5f * eps;
  const float pos_scale = (amg && a.step == 0) ? half : eps;
  const uint32_t S = (uint32_t)D, m = (S + 1) >> 1;

  // Loads of the evaluation point theta (SGLD, OBABO) or theta + scale M^-1 p (SGHMC,
  // AMAGOLD).
  const int q4 = 4 * ((threadIdx.x & (kWave - 1)) % LPR);
  float4 th[CPL];
  load_theta<LPR, CPL>(g_theta, D, th);
  float4 pe[CPL];
  if (shift && !resample) load_theta<LPR, CPL>(g_mom, D, pe);

  // Minibatch indices: (dkey', sub) = split(dkey); k1, k2 = split(sub).
  Key dnext, dsub;
  split2_uniform(dkey0, dnext, dsub);
  RowSource src;
  src.idx = nullptr;
  src.draw = 1;
  split2_uniform(dsub, src.k1, src.k2);
  src.n = (uint32_t)ch.n;
  src.span = (uint32_t)ch.N;
  src.mult = randint_mult(src.span);
  src.magic = randint_magic(src.span);
  src.rows = ch.N;

  float4 acc[CPL];
#pragma unroll
  for (int k = 0; k < CPL; ++k) acc[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  float lik_acc = 0.0f;
  int r0, r1, b0, b1;
  wave_rows(ch.n, ch.nblocks, bchain, r0, r1, b0, b1);
  // The step's noise: thread t owns the pairs jp = t + kNT h (h < NP, jp < m) of elements
  // jp and jp + m, which share one Threefry block. xr: the resampled momentum of the same
  // elements.
  Key knext;
  float xi[NP][2], xr[NP][2];
  accumulate_rows<LPR, CPL>(
      to_global(ch.X), ch.ldx, to_global(ch.y), D4, src, r0, r1, th, a.L, acc, lik_acc, lds.lik,
      b0, [&] {
        // Noise key of this step. OBABO: (key', s1, s2) = split(key, 3) at both launches of
        // a leapfrog step; the even one draws from s1, the odd one from s2 and stores key'.
        Key leaf;
        if (ob) {
          Key k0, s1, s2;
          split3(key0, k0, s1, s2);
          leaf = split_key(sub ? s2 : s1, 1, 0);
          knext = sub ? k0 : key0;
        } else {
          Key key_noise = key0, ksub;
          if (resample) {
            // momentum of this iteration: p = sqrt_mass * xi, drawn before the step's noise
            split2_uniform(key0, key_noise, ksub);
            const Key rleaf = split_key(ksub, 1, 0);
#pragma unroll
            for (int h = 0; h < NP; ++h) {
              const uint32_t jp = threadIdx.x + kNT * h;
              if (jp < m) {
                uint32_t w0, w1;
                bits_pair(rleaf, S, jp, w0, w1);
                xr[h][0] = bits_to_normal(w0);
                lds.p[jp] = a.sqrt_mass ? g_sqrt_mass[jp] * xr[h][0] : xr[h][0];
                if (jp + m < S) {
                  xr[h][1] = bits_to_normal(w1);
                  lds.p[jp + m] = a.sqrt_mass ? g_sqrt_mass[jp + m] * xr[h][1] : xr[h][1];
                }
              }
            }
          }
          split2_uniform(key_noise, knext, ksub);
          leaf = split_key(ksub, 1, 0);
        }
#pragma unroll
        for (int h = 0; h < NP; ++h) {
          const uint32_t jp = threadIdx.x + kNT * h;
          xi[h][0] = xi[h][1] = 0.0f;
          if (jp < m) {
            uint32_t w0, w1;
            bits_pair(leaf, S, jp, w0, w1);
            xi[h][0] = bits_to_normal(w0);
            xi[h][1] = bits_to_normal(w1);
          }
        }
        if (resample) {
          lds_sync();
#pragma unroll
          for (int k = 0; k < CPL; ++k) {
            float e[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const int c = q4 + 4 * LPR * k + t;
              e[t] = c < D ? lds.p[c] : 0.0f;
            }
            pe[k] = make_float4(e[0], e[1], e[2], e[3]);
          }
        }
        if (shift) {
#pragma unroll
          for (int k = 0; k < CPL; ++k) {
            const float p[4] = {pe[k].x, pe[k].y, pe[k].z, pe[k].w};
            float v[4] = {th[k].x, th[k].y, th[k].z, th[k].w};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const int c = q4 + 4 * LPR * k + t;
              if (c < D) {
                const float s = a.inv_mass ? g_inv_mass[c] * p[t] : p[t];
                v[t] = v[t] + pos_scale * s;
              }
            }
            th[k] = make_float4(v[0], v[1], v[2], v[3]);
          }
        }
      });
  // Block record: column sums, then the block's lik sum and its lik sum of squared
  // deviations about the block mean (combined into var(lik) by the last block). A chain of
  // one block keeps its record in LDS.
  // The two column sums of a noise pair lie side by side in the record and are written
  // and read by one 8-byte access each (two 4-byte ones where the caller's record buffer
  // is not 8-byte aligned).
  const int stride = 4 * D4 + 2;
  const bool single = ch.nblocks == 1;
  const bool wide = ((uintptr_t)ch.partial & 7) == 0;
  gfloat* mine = g_partial + (int64_t)bchain * stride;
  const float ls = block_reduce<LPR, CPL>(acc, lik_acc, D4, lds.cols, lds.small);
  float s[NP][2];
#pragma unroll
  for (int h = 0; h < NP; ++h) {
    const uint32_t jp = threadIdx.x + kNT * h;
    s[h][0] = s[h][1] = 0.0f;
    if (jp < m) {
      s[h][0] = col_sum(lds.cols, D4, jp);
      if (jp + m < S) s[h][1] = col_sum(lds.cols, D4, jp + m);
      if (!single) {
        if (wide) {
          publish2(mine + 2 * jp, s[h][0], s[h][1]);
        } else {
          publish(mine + 2 * jp, s[h][0]);
          publish(mine + 2 * jp + 1, s[h][1]);
        }
      }
    }
  }
  const int cnt = b1 - b0;
  float* slot1 = lds.small + kWaves;
  if (ch.var) {
    const float mb = cnt > 0 ? ls / (float)cnt : 0.0f;
    float s2 = 0.0f;
    for (int j = threadIdx.x; j < cnt; j += kNT) {
      const float d = lds.lik[j] - mb;
      s2 += d * d;
    }
    put_slot(slot1, s2);
  }
  if (ch.lik)
    for (int j = threadIdx.x; j < cnt; j += kNT) g_lik[b0 + j] = lds.lik[j];
  lds_sync();
  const float m2 = ch.var ? slot_sum(slot1) : 0.0f;
  if (!single && threadIdx.x == 0) {
    publish(mine + 4 * D4, ls);
    publish(mine + 4 * D4 + 1, m2);
  }
  // The state of the owned elements (the chain's other blocks only read it).
  float wv[NP][2], pv[NP][2], imv[NP][2], smv[NP][2], vv[NP][2];
#pragma unroll
  for (int h = 0; h < NP; ++h) {
    const uint32_t jp = threadIdx.x + kNT * h;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t j = e && jp + m < S ? jp + m : jp;
      const bool in = jp < m;
      wv[h][e] = in ? g_theta[j] : 0.0f;
      pv[h][e] = (in && has_mom && !resample) ? g_mom[j] : 0.0f;
      imv[h][e] = (in && has_mom && a.inv_mass) ? g_inv_mass[j] : 1.0f;
      smv[h][e] = (in && (resample || amg || ob) && a.sqrt_mass) ? g_sqrt_mass[j] : 1.0f;
      vv[h][e] = (in && rms) ? g_v[j] : 0.0f;
    }
  }
  if (!single && !arrive_last(ch.counter, ch.nblocks, &lds.flag)) return;

  // ---- last block of this chain: potential, gradient and the state update ----
  const bool last_step = !has_mom || a.step == launches - 1;
  // Every block of this chain has read the iteration counter. The last chain of the launch
  // to get here advances it (read by the next launch), on a wavefront that does not wait
  // for it.
  if (a.advance >= 0 && threadIdx.x == kNT - kWave) {
    const unsigned prev = atomicAdd(a.done, 1u);
    if (prev == (unsigned)a.nchains - 1) {
      atomicExch(a.done, 0u);
      if (last_step && a.advance) atomicAdd(a.iter, 1);
    }
  }
  const int nb = ch.nblocks;
  const float c = (float)(-ch.N) / (float)ch.n;
  const int per_block = (ch.n + nb - 1) / nb;
  float rec_ls = 0.0f, rec_m2 = 0.0f;
  if (single) {
    if (threadIdx.x == 0) {
      rec_ls = ls;
      rec_m2 = m2;
    }
  } else if (threadIdx.x < nb) {
    rec_ls = consume(g_partial + (int64_t)threadIdx.x * stride + 4 * D4);
    if (ch.var) rec_m2 = consume(g_partial + (int64_t)threadIdx.x * stride + 4 * D4 + 1);
  }
  // Column sums over the records, in block order; with more records than one round of
  // loads takes and threads to spare (m <= kNT / 2), in `parts` runs of blocks whose sums
  // are then added in order.
  constexpr bool kParts = 4 * LPR * CPL <= kNT;  // m <= kNT / 2
  if (single) {
    // the sum over one record starts from +0
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      s[h][0] = 0.0f + s[h][0];
      s[h][1] = 0.0f + s[h][1];
    }
  } else if (kParts && wide && nb > 16) {
    const int mp = m <= kNT / 4 ? kNT / 4 : kNT / 2;
    const int parts = kNT / mp, part = threadIdx.x / mp, jl = threadIdx.x % mp;
    const int per = (nb + parts - 1) / parts;
    float p0 = 0.0f, p1 = 0.0f;
    if (jl < (int)m)
      sum_pairs<16>(g_partial + 2 * jl, stride, part * per, min(nb, part * per + per), p0, p1);
    lds.cols[2 * threadIdx.x] = p0;
    lds.cols[2 * threadIdx.x + 1] = p1;
    lds_sync();
    s[0][0] = s[0][1] = 0.0f;
    if (threadIdx.x < mp)
      for (int k = 0; k < parts; ++k) {
        s[0][0] += lds.cols[2 * (k * mp + threadIdx.x)];
        s[0][1] += lds.cols[2 * (k * mp + threadIdx.x) + 1];
      }
  } else {
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      const uint32_t jp = threadIdx.x + kNT * h;
      if (jp >= m) break;
      gcfloat* p = g_partial + 2 * jp;
      // (the row buffers of CPL > 1 leave the registers for 32 records at their occupancy)
      if (wide) sum_pairs<(CPL > 1 ? 32 : 16)>(p, stride, 0, nb, s[h][0], s[h][1]);
      else sum_strided2(p, p + 1, stride, nb, s[h][0], s[h][1]);
    }
  }
  float sl = rec_ls;
  for (int b = threadIdx.x + kNT; b < nb; b += kNT)
    sl += consume(g_partial + (int64_t)b * stride + 4 * D4);
  put_slot(lds.small, sl);

  // AMAGOLD and SGGMC samples are saved after the Metropolis-Hastings test, not here.
  const int slot = (a.save_slot && !amg && !ob_mh) ? a.save_slot[it] : -1;
  const float Tn = ch.temperature;
  // obabo O-step coefficients (integrator.py:192-200): sqrt(exp(-f eps)) and
  // sqrt((1 - exp(-f eps)) T), float32.
  float ob_decay = 0.0f, ob_noise = 0.0f;
  if (ob) {
    const float perm = expf((-a.friction) * eps);
    ob_noise = sqrtf((1.0f - perm) * Tn);
    ob_decay = sqrtf(perm);
  }
  // reversible_leapfrog momentum coefficients (integrator.py:420-437), float32.
  const float ef = eps * a.friction;
  const float am_decay = 1.0f - ef;
  const float am_rescale = 1.0f / (1.0f + ef);
  const float am_noise = sqrtf(a.four_friction * eps);
  gfloat* g_theta_old = to_global(ch.theta_old);
  gfloat* g_mom_old = to_global(ch.mom_old);
  float edot = 0.0f;

  float lp = 0.0f;
#pragma unroll
  for (int h = 0; h < NP; ++h) {
    const uint32_t jp = threadIdx.x + kNT * h;
    if (jp >= m) break;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (e && jp + m >= S) break;
      const uint32_t j = e ? jp + m : jp;
      const float x = xi[h][e];
      float wj = wv[h][e];
      float p = 0.0f, sm = 0.0f;
      if (has_mom) {
        if (resample) p = a.sqrt_mass ? smv[h][e] * xr[h][e] : xr[h][e];
        else p = pv[h][e];
        sm = a.inv_mass ? imv[h][e] * p : p;
        if (shift) wj = wj + pos_scale * sm;  // evaluation point
      }
      float g = c * s[h][e];
      if (a.pr.has_prior) {
        g = g + wj * a.pr.inv_var;
        lp += (a.pr.log_norm + (wj * wj) * a.pr.inv_var) / -2.0f;
      }
      g = g / a.pot_temperature;
      float wn;
      if (!has_mom) {
        const float sg = (-eps) * g;
        const float sn = sqrtf((2.0f * Tn) * eps) * x;
        if (rms) {
          const float vn = a.alpha * vv[h][e] + (1.0f - a.alpha) * (g * g);
          g_v[j] = vn;
          const float G = 1.0f / (a.lmbd + sqrtf(vn));
          wn = wj + ((0.0f + G * sg) + sqrtf(G) * sn);
        } else {
          wn = wj + (sg + sn);
        }
      } else if (hmc) {
        const float C = a.friction;
        float pn = p + ((-eps) * C) * sm;
        pn = pn + (-eps) * g;
        pn = pn + C * (sqrtf(2.0f * eps) * x);
        g_mom[j] = pn;
        wn = wj;
      } else if (ob) {
        if (sub == 0) {
          // O: p1 = decay p + noise (M^{1/2} xi); B: p2 = (-eps/2) g + p1;
          // A: theta += eps M^-1 p2 (integrator.py:214-238).
          const float p1 = ob_decay * p + ob_noise * (smv[h][e] * x);
          edot += p1 * (imv[h][e] * p1);
          const float p2 = (-half) * g + p1;
          if (ob_mh && a.step == 0) {
            g_theta_old[j] = wv[h][e];
            g_mom_old[j] = p;
          }
          g_mom[j] = p2;
          wn = wj + eps * (imv[h][e] * p2);
        } else {
          // B: p3 = (-eps/2) g + p2; O with the second noise (integrator.py:244-262).
          const float p3 = (-half) * g + p;
          edot += p3 * (imv[h][e] * p3);
          g_mom[j] = ob_decay * p3 + ob_noise * (smv[h][e] * x);
          wn = wj;
        }
      } else {
        // p' = (((1 - eps f) p + (-eps) g) + sqrt(4 f eps) (M^{1/2} xi)) / (1 + eps f);
        // energy term (p + p') . (M^-1 g); final half position step after the last.
        const float noise = am_noise * (smv[h][e] * x);
        const float pn = am_rescale * ((am_decay * p + (-eps) * g) + noise);
        edot += (p + pn) * (imv[h][e] * g);
        if (a.step == 0) {
          g_theta_old[j] = wv[h][e];
          g_mom_old[j] = p;
        }
        g_mom[j] = pn;
        wn = last_step ? wj + half * (imv[h][e] * pn) : wj;
      }
      g_theta[j] = wn;
      if (slot >= 0 && last_step && ch.samples) g_samples[(int64_t)slot * D + j] = wn;
    }
  }
  lds_sync();  // the lik sums of the records
  const float mean = slot_sum(lds.small) / (float)ch.n;
  // var(lik) = (sum_b M2_b + cnt_b (mean_b - mean)^2) / n  (pairwise/Chan combination)
  if (ch.var) {
    float t = 0.0f;
    for (int b = threadIdx.x; b < nb; b += kNT) {
      const int lo = min(ch.n, b * per_block);
      const int k = min(ch.n, lo + per_block) - lo;
      if (k > 0) {
        const bool held = b < kNT;
        const float ls_b = held ? rec_ls : consume(g_partial + (int64_t)b * stride + 4 * D4);
        const float m2_b = held ? rec_m2 : consume(g_partial + (int64_t)b * stride + 4 * D4 + 1);
        const float d = ls_b / (float)k - mean;
        t += m2_b + (float)k * (d * d);
      }
    }
    put_slot(lds.small + kWaves, t);
  }
  put_slot(lds.small + 2 * kWaves, lp);
  if (amg || ob) put_slot(lds.small + 3 * kWaves, edot);
  lds_sync();
  if (threadIdx.x == 0) {
    lp = slot_sum(lds.small + 2 * kWaves);
    if (amg || ob) edot = slot_sum(lds.small + 3 * kWaves);
    if (amg) ch.energy[0] = half * edot + (a.step == 0 ? 0.0f : ch.energy[0]);
    if (ob) ch.energy[sub] = ch.energy[sub] + 0.5f * edot;
    const float Uc = ((float)(-ch.N) * mean - lp) / a.pot_temperature;
    // OBABO's potential is the mean of the step's two evaluations.
    float Uk = Uc;
    if (ob && sub) Uk = 0.5f * (ch.U[0] + Uc);
    if (ob_mh && a.step == 0) ch.energy[2] = ch.U[0];
    ch.U[0] = Uk;
    if (slot >= 0 && last_step && ch.samples_U) ch.samples_U[slot] = Uk;
    if (ch.var) ch.var[0] = slot_sum(lds.small + kWaves) / (float)ch.n;
    store_key(ch.key, knext);
    store_key(ch.dkey, dnext);
  }
}

// ---- resident loop: one single-block SGLD chain, many iterations on chip ----
// For chains of D <= 4 LPR (one float4 chunk per lane of a row segment) and minibatches
// of at most 256 rows (one 64-row chunk per wavefront), the chain's state stays on chip
// for the whole launch: theta in LDS (and its owner threads' registers), the keys in
// registers, the wavefronts' column partials in LDS. The step's noise is drawn one
// iteration ahead, beside the previous update; the minibatch of the next evaluation (its
// indices depend only on the data key) is drawn and its rows loaded right after this
// evaluation's row groups are consumed, so their latency overlaps the reduction and the
// update. The arithmetic
// is fused_body's for a chain of one block, in the same order (row groups, reductions,
// the SGLD / rms_prop update, U, var), so both give the same bits.
template <int LPR, int MODE>
__device__ __forceinline__ void resident_loop(const FusedArgs& a, const sgmc_glm_chain& ch,
                                              int iterations, float* lds_cols, float* lds_small,
                                              float* lds_lik, float* th_lds, float* eps_lds,
                                              int* slot_lds, uint32_t* kp, float* xis) {
  constexpr int CPL = 1;
  using RG = RowGroup<LPR, CPL>;
  constexpr int G = (kWave / LPR) * RG::U;  // rows per group
  constexpr int NG = kWave / G;             // groups of a 64-row chunk
  constexpr int kSegs = kWave / LPR;         // row segments of a wavefront
  constexpr int mode = MODE;
  const bool rms = mode == SGMC_MODE_SGLD_RMS;
  const int D = ch.D, D4 = (D + 3) >> 2, n = ch.n;
  gfloat* g_theta = to_global(ch.theta);
  gfloat* g_v = to_global(ch.v);
  gfloat* g_samples = to_global(ch.samples);
  const int it0 = a.iter[0];
  const int wv = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  // Thread jp < m owns the noise pair (jp, jp + m), as in fused_body's update loop.
  const uint32_t S = (uint32_t)D, m = (S + 1) >> 1;
  const uint32_t jp = threadIdx.x;
  const bool own = jp < m;
  const bool two = own && jp + m < S;
  const uint32_t jj[2] = {jp, two ? jp + m : jp};
  float w[2] = {0.0f, 0.0f}, v[2] = {0.0f, 0.0f};
  if (own) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[h] = g_theta[jj[h]];
      if (rms) v[h] = g_v[jj[h]];
    }
  }
  for (int c = threadIdx.x; c < 4 * LPR; c += kNT) th_lds[c] = c < D ? g_theta[c] : 0.0f;
  int r0, r1, b0, b1;
  wave_rows(n, 1, 0, r0, r1, b0, b1);
  const int ng = r0 < r1 ? (r1 - r0 + G - 1) / G : 0;  // wavefront-uniform
  RowSource src;
  src.idx = nullptr;
  src.draw = 1;
  src.n = (uint32_t)n;
  src.span = (uint32_t)ch.N;
  src.mult = randint_mult(src.span);
  src.magic = randint_magic(src.span);
  src.rows = ch.N;
  RG buf[NG];
  // The theta-independent key work runs ahead of its use, after the reduction barrier
  // (beside wavefront 0's update), handed over through LDS (kp, xis; slot = iteration
  // parity) across the loop's barriers. With key_{i+1}, ks_i = split(key_i), leaf_i =
  // split_key(ks_i, 1, 0) (the noise of iteration i), d_{i+1}, dsub_i = split(d_i) and
  // (k1_i, k2_i) = split(dsub_i) (the minibatch of iteration i), at iteration t:
  // - wavefront 3 runs one Threefry block per lane for all key steps at once: lanes 0-1
  //   split(key_{t+3}), lane 2 split_key(ks_{t+2}), lanes 3-4 split(d_{t+3}), lanes 5-6
  //   split(dsub_{t+2}); leaf_{t+2} goes to kp[2 slot ..], (k1, k2)_{t+2} to
  //   kp[4 + 4 slot ..], the chain states stay in its registers;
  // - wavefront 2 draws the normals of iteration t + 1 (lane l: word l / 32 of noise
  //   pair l % 32) into xis[64 slot' + 2 jp + h].
  // kp[12 ..]: the keys after the launch's last iteration.
  auto put_key = [&](int at, Key k) { kp[at] = k.k0; kp[at + 1] = k.k1; };
  auto get_key = [&](int at) { return Key{kp[at], kp[at + 1]}; };
  // the wavefront's rows of a minibatch with randint keys (k1, k2) into buf; a wavefront
  // of at most 32 rows draws their two randint words on the two lane halves (lanes 0-31
  // the words of k1, lanes 32-63 those of k2), one Threefry block per lane
  const bool halves = r1 - r0 <= kWave / 2;
  auto draw_rows = [&](Key k1, Key k2) {
    src.k1 = k1;
    src.k2 = k2;
    int rid = -1;
    if (halves) {
      const int rr = lane & (kWave / 2 - 1);
      const Key kk = lane < kWave / 2 ? src.k1 : src.k2;
      const uint32_t word = bits_word(kk, src.n, (uint32_t)(r0 + rr));
      const uint32_t lo = (uint32_t)__shfl((int)word, rr + kWave / 2, kWave);
      if (lane < kWave / 2 && r0 + rr < r1) {
        const int64_t r = (int64_t)randint_offset(word, lo, src.span, src.mult, src.magic);
        if (r >= 0 && r < src.rows) rid = (int)r;
      }
    } else if (r0 < r1) {
      rid = chunk_rows(src, r0, r1);
    }
#pragma unroll
    for (int gi = 0; gi < NG; ++gi)
      if (gi < ng) load_group<LPR, CPL>(to_global(ch.X), ch.ldx, to_global(ch.y), D4, gi * G, rid,
                                        buf[gi]);
  };
  // wavefront 3's chain states at iteration t: key_{t+3}, ks_{t+2}, d_{t+3}, dsub_{t+2}
  Key kc, ksn, dc, dsn;
  {
    // keys of iterations 0 to 2 (every thread; uniform values)
    Key key1, key2, ks0, ks1, d1, d2, ds0, ds1, k1, k2, k1n, k2n;
    split2_uniform(load_key(ch.key), key1, ks0);
    split2_uniform(key1, key2, ks1);
    split2_uniform(key2, kc, ksn);
    const Key leaf0 = split_key(ks0, 1, 0);
    const Key leaf1 = split_key(ks1, 1, 0);
    split2_uniform(load_key(ch.dkey), d1, ds0);
    split2_uniform(d1, d2, ds1);
    split2_uniform(d2, dc, dsn);
    split2_uniform(ds0, k1, k2);
    split2_uniform(ds1, k1n, k2n);
    if (threadIdx.x == 0) {
      put_key(2, leaf1);
      put_key(8, k1n);
      put_key(10, k2n);
      // the keys after the launch (iterations >= 3: set again in the loop)
      put_key(12, iterations == 1 ? key1 : iterations == 2 ? key2 : kc);
      put_key(14, iterations == 1 ? d1 : iterations == 2 ? d2 : dc);
    }
    if (own) {  // the normals of iteration 0
      uint32_t wb0, wb1;
      bits_pair(leaf0, S, jp, wb0, wb1);
      xis[2 * jp] = bits_to_normal(wb0);
      if (two) xis[2 * jp + 1] = bits_to_normal(wb1);
    }
    draw_rows(k1, k2);
  }
  const float c = (float)(-ch.N) / (float)n;
  const float Tn = ch.temperature;
  float Uk = 0.0f;
  // Barriers inside the loop wait for LDS only (lds_sync): the next minibatch's row
  // loads stay in flight through the reduction and the update. The step sizes and save
  // slots come from LDS (a window of kResWindow iterations), so no global load has to be
  // waited on behind those row loads. An iteration has two barriers (the wavefronts'
  // reduction records, the new theta), four more where U or var(lik) is kept.
  for (int t = 0; t < iterations; ++t) {
    const int tw = t % kResWindow;
    if (tw == 0) {
      __syncthreads();
      for (int u = threadIdx.x; u < kResWindow; u += kNT) {
        const int iu = max(0, min(it0 + t + u, a.table_len - 1));
        eps_lds[u] = a.eps_table[iu];
        slot_lds[u] = a.save_slot ? a.save_slot[iu] : -1;
      }
      __syncthreads();
    }
    const float eps = eps_lds[tw];
    const int slot = slot_lds[tw];
    const int par = t & 1;
    float4 th[CPL];
    {
      const int q = (threadIdx.x & (kWave - 1)) % LPR;
      th[0] = make_float4(th_lds[4 * q], th_lds[4 * q + 1], th_lds[4 * q + 2], th_lds[4 * q + 3]);
    }
    float4 acc[CPL];
    acc[0] = make_float4(0.f, 0.f, 0.f, 0.f);
    float lik_acc = 0.0f;
#pragma unroll
    for (int gi = 0; gi < NG; ++gi)
      if (gi < ng) process_group<LPR, CPL>(buf[gi], r0 + gi * G, D4, th, a.L, acc, lik_acc, lds_lik, 0);
    if (t + 1 < iterations) draw_rows(get_key(4 + 4 * (par ^ 1)), get_key(6 + 4 * (par ^ 1)));
    // Every lane's column partials go to LDS unreduced (one barrier); each owner thread
    // then adds its two columns over the row segments in the order of block_reduce's
    // segment shuffles (pairs of segments, pairs of pairs, ...) and over the wavefronts
    // in block_reduce's order. The lik sum is only formed where U is kept.
    const bool want_u = (slot >= 0 && ch.samples_U) || t == iterations - 1;
    {
      reinterpret_cast<float4*>(lds_cols)[wv * kWave + lane] = acc[0];
      if (want_u) {
        const float lw = wave_sum(lik_acc);
        if (lane == 0) lds_small[wv] = lw;
      }
    }
    // the owners' terms that do not need the column sums, before the barrier: the prior
    // gradient and log density, the noise term
    float lp = 0.0f, pg[2] = {0.0f, 0.0f}, sn[2] = {0.0f, 0.0f};
    if (own) {
      const float nscale = sqrtf((2.0f * Tn) * eps);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h && !two) break;
        const float wj = w[h];
        if (a.pr.has_prior) {
          pg[h] = wj * a.pr.inv_var;
          lp += (a.pr.log_norm + (wj * wj) * a.pr.inv_var) / -2.0f;
        }
        sn[h] = nscale * xis[64 * par + 2 * jp + h];
      }
    }
    lds_sync();
    if (wv == 3) {  // every key step of this iteration in one Threefry block per lane
      Key k = kc;
      uint32_t x0 = lane & 1, x1 = (lane & 1) + 2u;  // lanes 0, 1: split(key_{t+3})
      if (lane == 2) {  // split_key(ks_{t+2}, 1, 0)
        k = ksn;
        x0 = 0u;
        x1 = 1u;
      } else if (lane == 3 || lane == 4) {  // split(d_{t+3})
        k = dc;
        x0 = lane - 3;
        x1 = lane - 1;
      } else if (lane >= 5) {  // lanes 5, 6: split(dsub_{t+2})
        k = dsn;
        x0 = (lane - 5) & 1;
        x1 = x0 + 2u;
      }
      threefry2x32(k.k0, k.k1, x0, x1);
      auto rl = [](uint32_t v, int src) {
        return (uint32_t)__builtin_amdgcn_readlane((int)v, src);
      };
      if (t + 3 == iterations && lane == 0) {
        put_key(12, kc);
        put_key(14, dc);
      }
      if (lane == 0) {
        put_key(2 * par, Key{rl(x0, 2), rl(x1, 2)});
        put_key(4 + 4 * par, Key{rl(x0, 5), rl(x0, 6)});
        put_key(6 + 4 * par, Key{rl(x1, 5), rl(x1, 6)});
      }
      kc = Key{rl(x0, 0), rl(x0, 1)};
      ksn = Key{rl(x1, 0), rl(x1, 1)};
      dc = Key{rl(x0, 3), rl(x0, 4)};
      dsn = Key{rl(x1, 3), rl(x1, 4)};
    } else if (wv == 2 && t + 1 < iterations) {  // normals of iteration t + 1
      const uint32_t q = (uint32_t)lane & 31u, h = (uint32_t)lane >> 5;
      if (q < m && (h == 0 || q + m < S)) {
        uint32_t wb0, wb1;
        bits_pair(get_key(2 * (par ^ 1)), S, q, wb0, wb1);
        xis[64 * (par ^ 1) + 2 * q + h] = bits_to_normal(h ? wb1 : wb0);
      }
    }
    if (own) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h && !two) break;
        const uint32_t j = jj[h];
        float sc = 0.0f;
#pragma unroll
        for (int ww = 0; ww < kWaves; ++ww) {
          float sv[kSegs];
#pragma unroll
          for (int sg = 0; sg < kSegs; ++sg) sv[sg] = lds_cols[(ww * kWave + sg * LPR) * 4 + j];
#pragma unroll
          for (int w2 = 1; w2 < kSegs; w2 <<= 1)
#pragma unroll
            for (int i = 0; i < kSegs; i += 2 * w2) sv[i] = sv[i] + sv[i + w2];
          sc += sv[0];
        }
        const float wj = w[h];
        // one published record: the last block's sum over records starts from +0
        float g = c * (0.0f + sc);
        if (a.pr.has_prior) g = g + pg[h];
        if (a.pot_temperature != 1.0f) g = g / a.pot_temperature;  // x / 1 is x
        const float sg = (-eps) * g;
        float wn;
        if (rms) {
          const float vn = a.alpha * v[h] + (1.0f - a.alpha) * (g * g);
          v[h] = vn;
          const float Gs = 1.0f / (a.lmbd + sqrtf(vn));
          wn = wj + ((0.0f + Gs * sg) + sqrtf(Gs) * sn[h]);
        } else {
          wn = wj + (sg + sn[h]);
        }
        w[h] = wn;
        th_lds[j] = wn;
        if (slot >= 0 && ch.samples) g_samples[(int64_t)slot * D + j] = wn;
      }
    }
    // U (and var(lik)) only where they are kept: a save slot or the last iteration
    const bool last = t == iterations - 1;
    if (want_u) {
      float ls = 0.0f;  // read before block_sum's barrier lets lds_small be reused
#pragma unroll
      for (int i = 0; i < kWaves; ++i) ls += lds_small[i];
      lp = block_sum<kNT, true>(lp, lds_small);
      // the block's lik sum is the only record: the sum over records is ls + 0
      const float mean = (ls + 0.0f) / (float)n;
      Uk = ((float)(-ch.N) * mean - lp) / a.pot_temperature;
      if (threadIdx.x == 0 && slot >= 0 && ch.samples_U) ch.samples_U[slot] = Uk;
      if (ch.var && last) {
        // var(lik) of the last evaluation, as fused_body forms it from one record
        const float mb = n > 0 ? ls / (float)n : 0.0f;
        float s2 = 0.0f;
        for (int jr = threadIdx.x; jr < n; jr += kNT) {
          const float d = lds_lik[jr] - mb;
          s2 += d * d;
        }
        const float m2 = block_sum<kNT, true>(s2, lds_small);
        float tv = 0.0f;
        if (threadIdx.x == 0 && n > 0) {
          const float d = ls / (float)n - mean;
          tv += m2 + (float)n * (d * d);
        }
        const float var_sum = block_sum<kNT, true>(tv, lds_small);
        if (threadIdx.x == 0) ch.var[0] = var_sum / (float)n;
      }
    }
    lds_sync();
  }
  if (own) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h && !two) break;
      g_theta[jj[h]] = w[h];
      if (rms) g_v[jj[h]] = v[h];
    }
  }
  if (threadIdx.x == 0) {
    ch.U[0] = Uk;
    store_key(ch.key, get_key(12));
    store_key(ch.dkey, get_key(14));
  }
}

// Many iterations in one launch for tables whose chains have one block each: block c
// runs chain c's iterations back to back (every leapfrog step of every iteration),
// reading its parameters and keys back from memory after a barrier, so no launch and
// no arrival counter separates two evaluations. The last chain to finish advances the
// iteration counter by the number of iterations.
template <int DCLASS, int MODE>
__global__ void __launch_bounds__(kNT) glm_loop_kernel(FusedArgs a, int iterations) {
  __shared__ FusedLds<MODE> lds;
  // The grid has one block per chain and every chain one block (sgmc_glm_check_table).
  const int chain = blockIdx.x;
  const sgmc_glm_chain ch = a.chains[chain];
  const int dc = DCLASS >= 0 ? DCLASS : ch.dclass;
  FusedArgs b = a;
  b.advance = -1;
  const int launches = MODE == SGMC_MODE_OBABO ? 2 * a.steps : a.steps;
  // SGLD chains of D <= 64 and minibatches of at most 256 rows without per-row
  // likelihood output run resident (block-uniform choice)
  bool resident = false;
  constexpr bool kResident = (DCLASS == 0 || DCLASS == 5 || DCLASS == 1) &&
                             (MODE == SGMC_MODE_SGLD || MODE == SGMC_MODE_SGLD_RMS);
  if constexpr (kResident) {
    __shared__ float res_th[64];
    __shared__ float res_eps[kResWindow];
    __shared__ int res_slot[kResWindow];
    __shared__ uint32_t res_kp[16];
    __shared__ float res_xi[128];
    resident = !ch.lik && ch.n <= kWaves * kWave;
    if (resident)
      resident_loop<DCLASS == 0 ? 4 : DCLASS == 5 ? 8 : 16, MODE>(
          a, ch, iterations, lds.cols, lds.small, lds.lik, res_th, res_eps, res_slot, res_kp,
          res_xi);
  }
  for (int t = 0; t < (resident ? 0 : iterations); ++t) {
    b.iter_offset = t;
    for (int st = 0; st < launches; ++st) {
      b.step = st;
      switch (dc) {
        case 0: fused_body<4, 1, MODE>(b, ch, 0, lds); break;
        case 1: fused_body<16, 1, MODE>(b, ch, 0, lds); break;
        case 5: fused_body<8, 1, MODE>(b, ch, 0, lds); break;
        case 6: fused_body<32, 1, MODE>(b, ch, 0, lds); break;
        case 2: fused_body<64, 1, MODE>(b, ch, 0, lds); break;
        case 3: fused_body<64, 2, MODE>(b, ch, 0, lds); break;
        default: fused_body<64, 4, MODE>(b, ch, 0, lds); break;
      }
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) {
    const unsigned prev = atomicAdd(a.done, 1u);
    if (prev == (unsigned)a.nchains - 1) {
      atomicExch(a.done, 0u);
      atomicAdd(a.iter, iterations);
    }
  }
}

template <int DCLASS, int MODE>
__global__ void __launch_bounds__(kNT) glm_fused_kernel(FusedArgs a) {
  __shared__ FusedLds<MODE> lds;
  // A uniform table maps blocks to chains arithmetically, which saves the dependent
  // load of the map before the chain descriptor can be read.
  // The block map and the chains' block ranges agree (sgmc_glm_check_table checks the
  // table on the host before it is uploaded), so every block belongs to a chain.
  const int chain = a.blocks_per_chain > 0 ? (int)blockIdx.x / a.blocks_per_chain
                                           : a.block_chain[blockIdx.x];
  // The chain descriptor is copied once: block-uniform, it lives in scalar registers
  // instead of being re-read after every barrier and atomic.
  const sgmc_glm_chain ch = a.chains[chain];
  const int bchain = blockIdx.x - ch.block_begin;
  const int dc = DCLASS >= 0 ? DCLASS : ch.dclass;
  switch (dc) {
    case 0: fused_body<4, 1, MODE>(a, ch, bchain, lds); break;
    case 1: fused_body<16, 1, MODE>(a, ch, bchain, lds); break;
    case 5: fused_body<8, 1, MODE>(a, ch, bchain, lds); break;
    case 6: fused_body<32, 1, MODE>(a, ch, bchain, lds); break;
    case 2: fused_body<64, 1, MODE>(a, ch, bchain, lds); break;
    case 3: fused_body<64, 2, MODE>(a, ch, bchain, lds); break;
    default: fused_body<64, 4, MODE>(a, ch, bchain, lds); break;
  }
}

// The fused kernels of a table: one D class (or -1, mixed, with the class switch per
// block), the mode compiled in. Reading the mode at run time costs scalar registers
// (112 spilled at D <= 256) and the finalizer's branches: a launch of 16 rms_prop chains
// (D = 100, n = 1000, 16 blocks each) 20.0 us, compiled in 17.7; 20 SGGMC chains (D = 90,
// n = 2000) 24.7 -> 22.1; 8 SGHMC chains (D = 1000, n = 4096) 40.9 -> 38.7.
template <int MODE>
void launch_fused(int dclass, int nblocks, hipStream_t s, const FusedArgs& a) {
  const dim3 grid(nblocks), block(kNT);
  switch (dclass) {
    case 0: hipLaunchKernelGGL((glm_fused_kernel<0, MODE>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((glm_fused_kernel<1, MODE>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((glm_fused_kernel<2, MODE>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((glm_fused_kernel<3, MODE>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((glm_fused_kernel<4, MODE>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((glm_fused_kernel<5, MODE>), grid, block, 0, s, a); break;
    case 6: hipLaunchKernelGGL((glm_fused_kernel<6, MODE>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((glm_fused_kernel<-1, MODE>), grid, block, 0, s, a); break;
  }
}

template <int MODE>
void launch_loop(int dclass, int nchains, int iterations, hipStream_t s, const FusedArgs& a) {
  const dim3 grid(nchains), block(kNT);
  switch (dclass) {
    case 0: hipLaunchKernelGGL((glm_loop_kernel<0, MODE>), grid, block, 0, s, a, iterations); break;
    case 1: hipLaunchKernelGGL((glm_loop_kernel<1, MODE>), grid, block, 0, s, a, iterations); break;
    case 2: hipLaunchKernelGGL((glm_loop_kernel<2, MODE>), grid, block, 0, s, a, iterations); break;
    case 3: hipLaunchKernelGGL((glm_loop_kernel<3, MODE>), grid, block, 0, s, a, iterations); break;
    case 4: hipLaunchKernelGGL((glm_loop_kernel<4, MODE>), grid, block, 0, s, a, iterations); break;
    case 5: hipLaunchKernelGGL((glm_loop_kernel<5, MODE>), grid, block, 0, s, a, iterations); break;
    case 6: hipLaunchKernelGGL((glm_loop_kernel<6, MODE>), grid, block, 0, s, a, iterations); break;
    default:
      hipLaunchKernelGGL((glm_loop_kernel<-1, MODE>), grid, block, 0, s, a, iterations);
      break;
  }
}

// Instantiated in glm_fused_<mode>.hip and glm_loop_<mode>.hip.
#define SGMC_EXTERN_FUSED(MODE) \
  extern template void launch_fused<MODE>(int, int, hipStream_t, const FusedArgs&);
#define SGMC_EXTERN_LOOP(MODE) \
  extern template void launch_loop<MODE>(int, int, int, hipStream_t, const FusedArgs&);
SGMC_EXTERN_FUSED(SGMC_MODE_SGLD)
SGMC_EXTERN_FUSED(SGMC_MODE_SGLD_RMS)
SGMC_EXTERN_FUSED(SGMC_MODE_SGHMC)
SGMC_EXTERN_FUSED(SGMC_MODE_AMAGOLD)
SGMC_EXTERN_FUSED(SGMC_MODE_OBABO)
SGMC_EXTERN_FUSED(SGMC_MODE_SGGMC)
SGMC_EXTERN_LOOP(SGMC_MODE_SGLD)
SGMC_EXTERN_LOOP(SGMC_MODE_SGLD_RMS)
SGMC_EXTERN_LOOP(SGMC_MODE_SGHMC)
SGMC_EXTERN_LOOP(SGMC_MODE_OBABO)

}  // namespace sgmc
