// Generalized-linear likelihood families on the device: stochastic potential and
// gradient (potential.py:159-214 under jax.value_and_grad, integrator.py:166, 593,
// 792), the full-data potential in FP64 (potential.py:219-293), and the fused
// multi-chain step that advances every chain of a chain table by one gradient
// evaluation per launch.
//
// Families, per observation (x_i, y_i), z_i = x_i . w:
//   linear-Gaussian  lik = (log(2 pi s^2) + (y - z)^2 / s^2) / (-2)   dlik/dz = (y - z) / s^2
//   logistic         lik = y z - log(1 + e^z)                          dlik/dz = y - sigmoid(z)
// Potential: U = (-N * mean(lik) - log_prior) / T;
//            grad U = ((-N / n) * sum_i dlik_i/dz x_i - grad log_prior) / T
// with the Gaussian prior log p = sum_j (log(2 pi s_p^2) + w_j^2 / s_p^2) / (-2).
#include <math.h>

#include <algorithm>
#include <mutex>

#include "glm_fused.h"

namespace sgmc {

// ---------------------------------------------------------------- plain path --

struct PotArgs {
  const float* X;
  const float* y;
  const int32_t* idx;
  const float* theta;
  float* out_U;
  float* out_grad;
  float* out_lik;
  float* out_var;
  float* partial;      // [nblocks][4*D4 + 2]
  unsigned* counter;   // [kPotCounters]: the launch's, then one per run of blocks
  int64_t ldx;
  int64_t N;
  int n, D, D4;
  int group;           // blocks per run of a two-level reduction, or 0
  Lik L;
  Prior pr;
  float temperature;
};

// Arrival counters of a potential launch.
constexpr int kPotCounters = 64;

// Blocks per run of the two-level reduction (0: one level). One level reads 32 records
// per memory round trip; beyond that the last block's serial sum outgrows the round trip and
// arrival that a second level adds (n = 40001, D = 301, 256 blocks: 121 us with one level
// of eight records per round trip, 20.8 with two).
static int pot_group(int nblocks) {
  if (nblocks <= 32) return 0;
  return std::max(16, (nblocks + kPotCounters - 2) / (kPotCounters - 1));
}

template <int LPR, int CPL>
__global__ void __launch_bounds__(kNT) glm_potential_kernel(PotArgs a) {
  __shared__ __attribute__((aligned(16))) float lds_cols[kWaves * kMaxD];
  __shared__ float lds_small[kWaves];
  __shared__ float lds_lik[kLdsRows];
  __shared__ int flag;
  float4 th[CPL];
  float4 acc[CPL];
#pragma unroll
  for (int k = 0; k < CPL; ++k) acc[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  float lik_acc = 0.0f;
  int r0, r1, b0, b1;
  wave_rows(a.n, gridDim.x, blockIdx.x, r0, r1, b0, b1);
  RowSource src{a.idx, 0, Key{0, 0}, Key{0, 0}, 0, 0, 0, 0, a.idx ? a.N : (int64_t)a.n};
  accumulate_rows<LPR, CPL>(to_global(a.X), a.ldx, to_global(a.y), a.D4, src, r0, r1, th, a.L,
                            acc, lik_acc, lds_lik, b0,
                            [&] { load_theta<LPR, CPL>(to_global(a.theta), a.D, th); });
  // Block record: column sums, the block's lik sum and its lik sum of squared deviations
  // about the block mean; per-row likelihoods go straight to out_lik. Columns 2j and
  // 2j + 1 are one 8-byte access (two 4-byte ones where the records are not 8-byte aligned).
  const int stride = 4 * a.D4 + 2;
  const int nb = gridDim.x;
  gfloat* part = to_global(a.partial);
  gfloat* mine = part + (int64_t)blockIdx.x * stride;
  const bool wide = ((uintptr_t)a.partial & 7) == 0;
  auto put2 = [&](gfloat* p, float s0, float s1) {
    if (wide) {
      publish2(p, s0, s1);
    } else {
      publish(p, s0);
      publish(p + 1, s1);
    }
  };
  const float ls = block_reduce<LPR, CPL>(acc, lik_acc, a.D4, lds_cols, lds_small);
  for (int j = threadIdx.x; j < 2 * a.D4; j += kNT)
    put2(mine + 2 * j, col_sum(lds_cols, a.D4, 2 * j), col_sum(lds_cols, a.D4, 2 * j + 1));
  const int cnt = b1 - b0;
  float m2 = 0.0f;
  if (a.out_var) {
    const float mb = cnt > 0 ? ls / (float)cnt : 0.0f;
    float s2 = 0.0f;
    for (int j = threadIdx.x; j < cnt; j += kNT) {
      const float d = lds_lik[j] - mb;
      s2 += d * d;
    }
    m2 = block_sum<kNT>(s2, lds_small);
  }
  if (threadIdx.x == 0) {
    publish(mine + 4 * a.D4, ls);
    publish(mine + 4 * a.D4 + 1, m2);
  }
  if (a.out_lik) {
    gfloat* lo = to_global(a.out_lik);
    for (int j = threadIdx.x; j < cnt; j += kNT) lo[b0 + j] = lds_lik[j];
  }
  // Sums columns 2j, 2j + 1 over records 0 .. count - 1 of a run, `step` records apart.
  auto sum2 = [&](gcfloat* p, int64_t step, int count, float& s0, float& s1) {
    if (wide) sum_pairs<32>(p, step, 0, count, s0, s1);
    else sum_strided2(p, p + 1, step, count, s0, s1);
  };
  // Many blocks reduce in two levels: the last block of each run of `group` blocks sums the
  // run's columns into the run's first record, the last of those sums the runs.
  const int runs = a.group ? (nb + a.group - 1) / a.group : nb;
  const int64_t step = a.group ? (int64_t)a.group * stride : stride;
  if (a.group) {
    const int run = blockIdx.x / a.group, first = run * a.group;
    const int members = min(a.group, nb - first);
    if (!arrive_last(a.counter + 1 + run, members, &flag)) return;
    gfloat* p = part + (int64_t)first * stride;
    for (int j = threadIdx.x; j < 2 * a.D4; j += kNT) {
      float s0, s1;
      sum2(p + 2 * j, stride, members, s0, s1);
      put2(p + 2 * j, s0, s1);
    }
  }
  if (!arrive_last(a.counter, runs, &flag)) return;

  // Last block: combine the block records, add the prior, scale.
  const float c = (float)(-a.N) / (float)a.n;
  float sl = 0.0f;
  for (int b = threadIdx.x; b < nb; b += kNT) sl += consume(part + (int64_t)b * stride + 4 * a.D4);
  float lp = 0.0f;
  for (int j2 = threadIdx.x; j2 < 2 * a.D4; j2 += kNT) {
    float s[2];
    sum2(part + 2 * j2, step, runs, s[0], s[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int j = 2 * j2 + e;
      if (j >= a.D) break;
      const float wj = a.theta[j];
      float g = c * s[e];
      if (a.pr.has_prior) {
        g = g + wj * a.pr.inv_var;
        lp += (a.pr.log_norm + (wj * wj) * a.pr.inv_var) / -2.0f;
      }
      a.out_grad[j] = g / a.temperature;
    }
  }
  const float sumlik = block_sum<kNT>(sl, lds_small);
  const float mean = sumlik / (float)a.n;
  lp = block_sum<kNT>(lp, lds_small);
  if (threadIdx.x == 0) a.out_U[0] = ((float)(-a.N) * mean - lp) / a.temperature;
  if (a.out_var) {
    // var(lik) = (sum_b M2_b + cnt_b (mean_b - mean)^2) / n  (pairwise/Chan combination)
    const int per_block = (a.n + nb - 1) / nb;
    float t = 0.0f;
    for (int b = threadIdx.x; b < nb; b += kNT) {
      const int lo = min(a.n, b * per_block);
      const int k = min(a.n, lo + per_block) - lo;
      if (k > 0) {
        const float d = consume(part + (int64_t)b * stride + 4 * a.D4) / (float)k - mean;
        t += consume(part + (int64_t)b * stride + 4 * a.D4 + 1) + (float)k * (d * d);
      }
    }
    t = block_sum<kNT>(t, lds_small);
    if (threadIdx.x == 0) a.out_var[0] = t / (float)a.n;
  }
}

// --------------------------------------------------------- full potential ----

struct FullArgs {
  const float* X;
  const float* y;
  const float* theta;
  double* out_U;
  double* partial;
  unsigned* counter;
  int64_t ldx;
  int64_t N;
  int D, D4;
  int rows_per_block;
  Lik L;
  Prior pr;
  double temperature;
};

// Streams the block's rows, each wavefront a contiguous quarter, one row group in flight
// ahead of the one being reduced (two register buffers); the rows of a group share one
// evaluation of the likelihood, row u on lane u of its segment. Bound by the read of X:
// N = 1e6, D = 512 in 488 blocks 342 us (6.0 TB/s), D = 100 72 us. (One row at a time with the
// likelihood on every lane spent about 210 us of vector issue per SIMD, not overlapped with
// its loads: 466 and 273 us in 977 blocks.) The row products are separate multiplies and
// adds: fused ones round differently, 2e-9 of a float64 potential of 11000 rows.
template <int LPR, int CPL>
__global__ void __launch_bounds__(kNT) glm_full_kernel(FullArgs a) {
  __shared__ double lds_d[kWaves];
  __shared__ int flag;
  constexpr int RPW = kWave / LPR;
  using RG = RowGroup<LPR, CPL>;
  constexpr int U = RG::U, G = RPW * U;
  const int lane = threadIdx.x & (kWave - 1);
  const int seg = lane / LPR, q = lane % LPR;
  float4 th[CPL];
  load_theta<LPR, CPL>(to_global(a.theta), a.D, th);
  const int64_t b0 = (int64_t)blockIdx.x * a.rows_per_block;
  const int rows = (int)min<int64_t>(a.N - b0, a.rows_per_block);
  gcfloat* X = to_global(a.X) + b0 * a.ldx;
  gcfloat* y = to_global(a.y) + b0;
  const int per = (rows + kWaves - 1) / kWaves;
  const int r0 = min(rows, (int)(threadIdx.x / kWave) * per), r1 = min(rows, r0 + per);
  double acc = 0.0;
  // rows r .. r + G - 1 of the wavefront (row r + u RPW + seg in slot u, -1 past its end)
  auto load = [&](int r, RG& g) {
    load_group<LPR, CPL>(X, a.ldx, y, a.D4, 0, r + lane < r1 ? r + lane : -1, g);
  };
  auto reduce = [&](RG& g) {
    float zq = 0.0f, yq = 0.0f;
    bool okq = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float t = 0.0f;
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        f4 x = g.x[u][k];
        // (a whole wavefront's rows read past their end as zero; shorter segments reload
        // their last chunk there)
        if (RPW > 1 && q + LPR * k >= a.D4) x = f4{0.f, 0.f, 0.f, 0.f};
        t += dot4(x, th[k]);
      }
      t = seg_sum<LPR>(t);
      zq = q == u ? t : zq;
      yq = q == u ? g.y[u] : yq;
      okq = q == u ? g.ok[u] : okq;
    }
    float lik, rr;
    row_lik(a.L, zq, yq, lik, rr);
    if (q < U && okq) acc += (double)lik;
  };
  if (r0 < r1) {
    RG ga, gb;
    load(r0, ga);
    for (int r = r0; r < r1; r += 2 * G) {
      load(r + G, gb);
      reduce(ga);
      load(r + 2 * G, ga);
      reduce(gb);
    }
  }
  const double bs = block_sum_d<kNT>(acc, lds_d);
  if (threadIdx.x == 0) publish(a.partial + blockIdx.x, bs);
  if (!arrive_last(a.counter, gridDim.x, &flag)) return;
  double tot = 0.0;
  for (int b = threadIdx.x; b < (int)gridDim.x; b += kNT) tot += consume(a.partial + b);
  tot = block_sum_d<kNT>(tot, lds_d);
  double lp = 0.0;
  if (a.pr.has_prior) {
    const double iv = (double)a.pr.inv_var;
    const double ln = (double)a.pr.log_norm;
    for (int j = threadIdx.x; j < a.D; j += kNT) {
      const double wj = (double)a.theta[j];
      lp += (ln + wj * wj * iv) / -2.0;
    }
  }
  lp = block_sum_d<kNT>(lp, lds_d);
  if (threadIdx.x == 0) a.out_U[0] = (-tot - lp) / a.temperature;
}

static int dclass_of(int D) {
  if (D <= 16) return 0;
  if (D <= 32) return 5;  // 8 lanes per row (added after 0-4: the numbers are labels)
  if (D <= 64) return 1;
  // 32 lanes per row, two rows per wavefront load: with 64 lanes (class 2) half of each
  // load is empty at D <= 128 (16 rms_prop chains, D = 100,
  // n = 1000, 16 blocks each, 15.7 -> 13.7 us per launch; in 2 blocks each 37.8 -> 25.3)
  if (D <= 128) return 6;
  if (D <= 256) return 2;
  if (D <= 512) return 3;
  return 4;
}

}  // namespace sgmc

using namespace sgmc;

namespace {

// Validates the arguments of a minibatch potential and launches its kernel with the
// block records at `partial` ([nblocks][4 ceil(D/4) + 2] floats) and the arrival counter
// at `counter` (zero before the launch; the last block resets it).
int launch_potential(const char* who, int family, const float* X, int64_t ldx, const float* y,
                     const int32_t* idx, int n, int64_t N, int D, const float* theta,
                     float sigma, int has_prior, float prior_scale, float temperature,
                     float* out_U, float* out_grad, float* out_lik, float* out_var,
                     float* partial, unsigned* counter, int group, int nblocks, void* stream) {
  SGMC_REQUIRE(X && y && theta && out_U && out_grad, SGMC_E_ARG, "%s: null pointer", who);
  SGMC_REQUIRE(family == SGMC_LIK_LINEAR_GAUSSIAN || family == SGMC_LIK_LOGISTIC, SGMC_E_ARG,
               "%s: unknown family %d", who, family);
  SGMC_REQUIRE(D >= 1 && D <= kMaxD, SGMC_E_ARG, "%s: D=%d outside [1, %d]", who, D, kMaxD);
  SGMC_REQUIRE(ldx % 4 == 0 && ldx >= 4 * ((D + 3) / 4), SGMC_E_ARG,
               "%s: ldx=%lld must be a multiple of 4 and >= D rounded up", who, (long long)ldx);
  SGMC_REQUIRE(((uintptr_t)X & 15) == 0, SGMC_E_ARG, "%s: X not 16B aligned", who);
  SGMC_REQUIRE(n >= 1 && N >= 1, SGMC_E_ARG, "%s: empty batch", who);
  SGMC_REQUIRE(nblocks >= 1 && (int64_t)nblocks * kLdsRows >= n, SGMC_E_ARG,
               "%s: nblocks must be >= 1 and >= n / %d", who, kLdsRows);
  SGMC_REQUIRE(temperature != 0.0f, SGMC_E_ARG, "%s: temperature is zero", who);
  PotArgs a;
  a.X = X;
  a.y = y;
  a.idx = idx;
  a.theta = theta;
  a.out_U = out_U;
  a.out_grad = out_grad;
  a.out_lik = out_lik;
  a.out_var = out_var;
  a.D = D;
  a.D4 = (D + 3) / 4;
  a.partial = partial;
  a.counter = counter;
  a.group = group;
  a.ldx = ldx;
  a.N = N;
  a.n = n;
  a.L = make_lik(family, sigma);
  a.pr = make_prior(has_prior, prior_scale);
  a.temperature = temperature;
  hipStream_t s = as_stream(stream);
  dim3 grid(nblocks), block(kNT);
  switch (dclass_of(D)) {
    case 0: hipLaunchKernelGGL((glm_potential_kernel<4, 1>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((glm_potential_kernel<16, 1>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((glm_potential_kernel<8, 1>), grid, block, 0, s, a); break;
    case 6: hipLaunchKernelGGL((glm_potential_kernel<32, 1>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((glm_potential_kernel<64, 1>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((glm_potential_kernel<64, 2>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((glm_potential_kernel<64, 4>), grid, block, 0, s, a); break;
  }
  return check_launch(who);
}

// ---- scratch of the no-allocation entry point (sgmc_glm_potential_noalloc) ----
// One 1 MiB array per GPU, held until the process ends: word 0 is the arrival counter
// (padded to 256 bytes, so it stays at one address whatever the call's size), the block
// records follow. Every call on a GPU shares that GPU's array; calls that overlap on one
// GPU race. The counter is zeroed when the array is first used on a device, and every
// call leaves it at zero (the potential's last block resets it); the records are
// written before they are read in every call.
constexpr int64_t kScratchFloats = 1 << 18;
constexpr int64_t kScratchCounterFloats = kPotCounters;
constexpr int64_t kScratchRecordFloats = kScratchFloats - kScratchCounterFloats;
constexpr int kScratchDevices = 64;
static __device__ __align__(256) float scratch[kScratchFloats];

__global__ void __launch_bounds__(kNT) zero_floats_kernel(float* p, int n) {
  const int i = blockIdx.x * kNT + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

std::mutex g_scratch_mu;
float* g_scratch[kScratchDevices] = {};

// Device address of the current device's scratch (the host-side name `scratch` is only
// a stand-in for it): looked up once per device with hipGetSymbolAddress, its counter
// zeroed on `stream` at that first use.
int scratch_of_current_device(void* stream, float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  SGMC_REQUIRE(e == hipSuccess, SGMC_E_HIP, "sgmc_glm_potential_noalloc: hipGetDevice: %s",
               hipGetErrorString(e));
  SGMC_REQUIRE(dev >= 0 && dev < kScratchDevices, SGMC_E_ARG,
               "sgmc_glm_potential_noalloc: device %d beyond %d", dev, kScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    float* p = nullptr;
    e = hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch));
    SGMC_REQUIRE(e == hipSuccess && p, SGMC_E_HIP,
                 "sgmc_glm_potential_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    hipLaunchKernelGGL(zero_floats_kernel, dim3(1), dim3(kNT), 0, as_stream(stream), p,
                       (int)kScratchCounterFloats);
    const int rc = check_launch("sgmc_glm_potential_noalloc: scratch set-up");
    if (rc != SGMC_OK) return rc;
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return SGMC_OK;
}

// ---- launches of one chain table ----
bool known_mode(int mode) { return mode >= SGMC_MODE_SGLD && mode <= SGMC_MODE_SGGMC; }

// Launches of one iteration: modes without leapfrog steps take one whatever `steps` says,
// OBABO modes two per leapfrog step.
int launches_of(const sgmc_glm_run& r) {
  if (r.mode == SGMC_MODE_SGLD || r.mode == SGMC_MODE_SGLD_RMS) return 1;
  return (r.mode == SGMC_MODE_OBABO || r.mode == SGMC_MODE_SGGMC) ? 2 * r.steps : r.steps;
}

// Modes that run many iterations in one launch: no Metropolis-Hastings test in between.
bool loop_mode(int mode) {
  return mode == SGMC_MODE_SGLD || mode == SGMC_MODE_SGLD_RMS || mode == SGMC_MODE_SGHMC ||
         mode == SGMC_MODE_OBABO;
}

int check_run(const char* who, const sgmc_glm_run& r) {
  SGMC_REQUIRE(r.chains && r.eps_table && r.iter && r.done, SGMC_E_ARG, "%s: null pointer", who);
  SGMC_REQUIRE(r.block_chain || (r.nchains > 0 && r.nblocks % r.nchains == 0), SGMC_E_ARG,
               "%s: without a block map nblocks must be a multiple of nchains", who);
  SGMC_REQUIRE(r.nchains >= 1 && r.nblocks >= r.nchains && r.table_len >= 1, SGMC_E_ARG,
               "%s: bad sizes", who);
  SGMC_REQUIRE(r.family == SGMC_LIK_LINEAR_GAUSSIAN || r.family == SGMC_LIK_LOGISTIC, SGMC_E_ARG,
               "%s: unknown family %d", who, r.family);
  SGMC_REQUIRE(known_mode(r.mode), SGMC_E_ARG, "%s: unknown mode %d", who, r.mode);
  SGMC_REQUIRE(r.steps >= 1, SGMC_E_ARG, "%s: steps %d", who, r.steps);
  SGMC_REQUIRE(r.pot_temperature != 0.0f, SGMC_E_ARG, "%s: temperature is zero", who);
  return SGMC_OK;
}

// The kernel arguments of a table's first launch of an iteration.
FusedArgs run_args(const sgmc_glm_run& r) {
  FusedArgs a;
  a.chains = r.chains;
  a.block_chain = r.block_chain;
  a.blocks_per_chain = r.block_chain ? 0 : r.nblocks / r.nchains;
  a.eps_table = r.eps_table;
  a.save_slot = r.save_slot;
  a.iter = r.iter;
  a.done = r.done;
  a.inv_mass = r.inv_mass;
  a.sqrt_mass = r.sqrt_mass;
  a.table_len = r.table_len;
  a.nchains = r.nchains;
  a.step = 0;
  a.steps = r.steps;
  a.friction = r.friction;
  a.four_friction = (float)(4.0 * (double)r.friction);
  a.alpha = r.alpha;
  a.lmbd = r.lmbd;
  a.L = make_lik(r.family, r.sigma);
  a.pr = make_prior(r.has_prior, r.prior_scale);
  a.pot_temperature = r.pot_temperature;
  a.advance = 1;
  a.iter_offset = 0;
  return a;
}

void launch_step(const sgmc_glm_run& r, const FusedArgs& a) {
  const int dc = r.uniform_dclass, nb = r.nblocks;
  hipStream_t s = as_stream(r.stream);
  switch (r.mode) {
    case SGMC_MODE_SGLD: launch_fused<SGMC_MODE_SGLD>(dc, nb, s, a); break;
    case SGMC_MODE_SGLD_RMS: launch_fused<SGMC_MODE_SGLD_RMS>(dc, nb, s, a); break;
    case SGMC_MODE_SGHMC: launch_fused<SGMC_MODE_SGHMC>(dc, nb, s, a); break;
    case SGMC_MODE_AMAGOLD: launch_fused<SGMC_MODE_AMAGOLD>(dc, nb, s, a); break;
    case SGMC_MODE_OBABO: launch_fused<SGMC_MODE_OBABO>(dc, nb, s, a); break;
    default: launch_fused<SGMC_MODE_SGGMC>(dc, nb, s, a); break;
  }
}

// `iterations` iterations of a table of one-block chains in one launch. Modes without
// leapfrog steps take one evaluation per iteration whatever `steps` says.
void launch_loop_mode(const sgmc_glm_run& r, int iterations, FusedArgs a) {
  if (r.mode != SGMC_MODE_SGHMC && r.mode != SGMC_MODE_OBABO) a.steps = 1;
  const int dc = r.uniform_dclass, n = r.nchains;
  hipStream_t s = as_stream(r.stream);
  switch (r.mode) {
    case SGMC_MODE_SGLD: launch_loop<SGMC_MODE_SGLD>(dc, n, iterations, s, a); break;
    case SGMC_MODE_SGLD_RMS: launch_loop<SGMC_MODE_SGLD_RMS>(dc, n, iterations, s, a); break;
    case SGMC_MODE_SGHMC: launch_loop<SGMC_MODE_SGHMC>(dc, n, iterations, s, a); break;
    default: launch_loop<SGMC_MODE_OBABO>(dc, n, iterations, s, a); break;
  }
}

// Tables whose launches one call takes in turn.
constexpr int kTogether = 64;

// Issues the operations of up to kTogether checked tables, one launch per table and turn.
int issue_runs(const sgmc_glm_run* runs, int nruns) {
  struct Cursor {
    int op = 0;
    int64_t at = 0;  // launches of the operation issued so far
  };
  Cursor cur[kTogether];
  for (bool any = true; any;) {
    any = false;
    for (int k = 0; k < nruns; ++k) {
      const sgmc_glm_run& r = runs[k];
      Cursor& c = cur[k];
      while (c.op < r.nops) {
        const int count = r.ops[2 * c.op + 1];
        const int64_t total = r.ops[2 * c.op] == SGMC_OP_ITERATIONS
                                  ? (int64_t)count * launches_of(r)
                                  : r.ops[2 * c.op] == SGMC_OP_LOOP ? (count > 0) : count;
        if (c.at < total) break;
        ++c.op;
        c.at = 0;
      }
      if (c.op == r.nops) continue;
      any = true;
      int rc;
      switch (r.ops[2 * c.op]) {
        case SGMC_OP_ITERATIONS: {
          FusedArgs a = run_args(r);
          a.step = (int)(c.at % launches_of(r));
          launch_step(r, a);
          rc = check_launch("sgmc_glm_fused_run");
          break;
        }
        case SGMC_OP_LOOP: {
          FusedArgs a = run_args(r);
          a.blocks_per_chain = 1;
          a.block_chain = nullptr;
          a.advance = -1;
          launch_loop_mode(r, r.ops[2 * c.op + 1], a);
          rc = check_launch("sgmc_glm_fused_run");
          break;
        }
        default:
          rc = sgmc_resgld_swap(r.chains, r.nchains, r.pairs, r.npairs, r.F, r.swap_every,
                                r.save_slot, r.table_len, r.iter, r.stream);
      }
      if (rc != SGMC_OK) return rc;
      ++c.at;
    }
  }
  return SGMC_OK;
}

}  // namespace

extern "C" {

int64_t sgmc_glm_workspace_floats(int n, int D, int nblocks) {
  const int D4 = (D + 3) / 4;
  (void)n;
  return (int64_t)nblocks * (4 * D4 + 2) + kPotCounters;
}

// One block per compute unit (two at 256 < D <= 512), each with at least one row group of its
// four wavefronts. n = 40001, D = 301: 19.3 us at 507 blocks, 20.8 at 256; n = 60000,
// D = 1000: 49.2 and 45.9; n = 20000, D = 100: 13.8 and 12.7; n = 60000, D = 64: 14.2 and
// 13.2. (256 rows per block, whatever the size: 87.5, 270.7, 38.2 and 63.3 us.) Never more
// records than the scratch of sgmc_glm_potential_noalloc holds (509 blocks at D = 512, 255 at
// D = 1024) unless the rows of a block need them.
int sgmc_glm_blocks(int n, int D) {
  const int held = (int)(kScratchRecordFloats / (4 * ((D + 3) / 4) + 2));
  const int blocks = std::min(D > 256 && D <= 512 ? 512 : 256, held);
  const int least = D <= 16 ? 256 : D <= 32 ? 128 : D <= 64 ? 64 : 32;
  const int rows = std::max(least, (int)(((int64_t)n + blocks - 1) / blocks));
  const int b = (int)(((int64_t)n + rows - 1) / rows);
  return std::max(b < 1 ? 1 : b, (int)(((int64_t)n + kLdsRows - 1) / kLdsRows));
}

int sgmc_glm_potential(int family, const float* X, int64_t ldx, const float* y,
                       const int32_t* idx, int n, int64_t N, int D, const float* theta,
                       float sigma, int has_prior, float prior_scale, float temperature,
                       float* out_U, float* out_grad, float* out_lik, float* out_var,
                       float* workspace, int64_t workspace_floats, int nblocks, void* stream) {
  SGMC_REQUIRE(workspace, SGMC_E_ARG, "sgmc_glm_potential: null workspace");
  SGMC_REQUIRE(D >= 1 && D <= kMaxD && nblocks >= 1, SGMC_E_ARG,
               "sgmc_glm_potential: D=%d outside [1, %d] or nblocks=%d", D, kMaxD, nblocks);
  const int64_t records = (int64_t)nblocks * (4 * ((D + 3) / 4) + 2);
  SGMC_REQUIRE(workspace_floats >= records + 4, SGMC_E_ARG,
               "sgmc_glm_potential: workspace too small");
  // a workspace with room for one counter only reduces in one level
  const int group = workspace_floats >= records + kPotCounters ? pot_group(nblocks) : 0;
  return launch_potential("sgmc_glm_potential", family, X, ldx, y, idx, n, N, D, theta, sigma,
                          has_prior, prior_scale, temperature, out_U, out_grad, out_lik,
                          out_var, workspace, reinterpret_cast<unsigned*>(workspace + records),
                          group, nblocks, stream);
}

int sgmc_glm_potential_noalloc(int family, const float* X, int64_t ldx, const float* y,
                               const int32_t* idx, int n, int64_t N, int D, const float* theta,
                               float sigma, int has_prior, float prior_scale, float temperature,
                               float* out_U, float* out_grad, float* out_lik, float* out_var,
                               int nblocks, void* stream) {
  SGMC_REQUIRE(D >= 1 && D <= kMaxD && nblocks >= 1, SGMC_E_ARG,
               "sgmc_glm_potential_noalloc: D=%d outside [1, %d] or nblocks=%d", D, kMaxD,
               nblocks);
  const int64_t records = (int64_t)nblocks * (4 * ((D + 3) / 4) + 2);
  SGMC_REQUIRE(records <= kScratchRecordFloats, SGMC_E_ARG,
               "sgmc_glm_potential_noalloc: %d blocks of D=%d need %lld record floats; the "
               "static scratch holds %lld (use sgmc_glm_potential with a workspace)",
               nblocks, D, (long long)records, (long long)kScratchRecordFloats);
  float* base = nullptr;
  const int rc = scratch_of_current_device(stream, &base);
  if (rc != SGMC_OK) return rc;
  return launch_potential("sgmc_glm_potential_noalloc", family, X, ldx, y, idx, n, N, D, theta,
                          sigma, has_prior, prior_scale, temperature, out_U, out_grad, out_lik,
                          out_var, base + kScratchCounterFloats,
                          reinterpret_cast<unsigned*>(base), pot_group(nblocks), nblocks, stream);
}

int64_t sgmc_glm_full_workspace_doubles(int64_t N, int rows_per_block) {
  return (N + rows_per_block - 1) / rows_per_block + 2;
}

int sgmc_glm_full_potential(int family, const float* X, int64_t ldx, const float* y, int64_t N,
                            int D, const float* theta, float sigma, int has_prior,
                            float prior_scale, double temperature, double* out_U,
                            double* workspace, int64_t workspace_doubles, int rows_per_block,
                            void* stream) {
  SGMC_REQUIRE(X && y && theta && out_U && workspace, SGMC_E_ARG,
               "sgmc_glm_full_potential: null pointer");
  SGMC_REQUIRE(family == SGMC_LIK_LINEAR_GAUSSIAN || family == SGMC_LIK_LOGISTIC, SGMC_E_ARG,
               "sgmc_glm_full_potential: unknown family %d", family);
  SGMC_REQUIRE(D >= 1 && D <= kMaxD, SGMC_E_ARG, "sgmc_glm_full_potential: D out of range");
  SGMC_REQUIRE(ldx % 4 == 0 && ldx >= 4 * ((D + 3) / 4), SGMC_E_ARG,
               "sgmc_glm_full_potential: bad ldx");
  SGMC_REQUIRE(((uintptr_t)X & 15) == 0, SGMC_E_ARG, "sgmc_glm_full_potential: X misaligned");
  SGMC_REQUIRE(N >= 1 && rows_per_block >= 1, SGMC_E_ARG, "sgmc_glm_full_potential: bad size");
  const int64_t nb = (N + rows_per_block - 1) / rows_per_block;
  SGMC_REQUIRE(nb <= 2147483647LL, SGMC_E_ARG, "sgmc_glm_full_potential: too many blocks");
  SGMC_REQUIRE(workspace_doubles >= sgmc_glm_full_workspace_doubles(N, rows_per_block),
               SGMC_E_ARG, "sgmc_glm_full_potential: workspace too small");
  SGMC_REQUIRE(temperature != 0.0, SGMC_E_ARG, "sgmc_glm_full_potential: temperature is zero");
  FullArgs a;
  a.X = X;
  a.y = y;
  a.theta = theta;
  a.out_U = out_U;
  a.partial = workspace;
  a.counter = reinterpret_cast<unsigned*>(workspace + nb);
  a.ldx = ldx;
  a.N = N;
  a.D = D;
  a.D4 = (D + 3) / 4;
  a.rows_per_block = rows_per_block;
  a.L = make_lik(family, sigma);
  a.pr = make_prior(has_prior, prior_scale);
  a.temperature = temperature;
  hipStream_t s = as_stream(stream);
  dim3 grid((unsigned)nb), block(kNT);
  switch (dclass_of(D)) {
    case 0: hipLaunchKernelGGL((glm_full_kernel<4, 1>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((glm_full_kernel<16, 1>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((glm_full_kernel<8, 1>), grid, block, 0, s, a); break;
    case 6: hipLaunchKernelGGL((glm_full_kernel<32, 1>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((glm_full_kernel<64, 1>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((glm_full_kernel<64, 2>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((glm_full_kernel<64, 4>), grid, block, 0, s, a); break;
  }
  return check_launch("sgmc_glm_full_potential");
}

int sgmc_glm_dclass(int D) { return dclass_of(D); }

int sgmc_glm_check_table(const sgmc_glm_chain* chains, int nchains, const int32_t* block_chain,
                         int nblocks, int loop) {
  SGMC_REQUIRE(chains && nchains >= 1, SGMC_E_ARG, "sgmc_glm_check_table: no chains");
  if (loop) {
    SGMC_REQUIRE(nblocks == nchains, SGMC_E_ARG,
                 "sgmc_glm_check_table: a loop launch has one block per chain");
  } else {
    SGMC_REQUIRE(nblocks >= nchains, SGMC_E_ARG, "sgmc_glm_check_table: %d blocks for %d chains",
                 nblocks, nchains);
    SGMC_REQUIRE(block_chain || nblocks % nchains == 0, SGMC_E_ARG,
                 "sgmc_glm_check_table: without a block map nblocks must be a multiple of "
                 "nchains");
  }
  const int per = !block_chain ? nblocks / nchains : 1;
  int64_t covered = 0;
  for (int c = 0; c < nchains; ++c) {
    const sgmc_glm_chain& ch = chains[c];
    SGMC_REQUIRE(ch.X && ch.y && ch.theta && ch.key && ch.dkey && ch.U && ch.partial &&
                     ch.counter,
                 SGMC_E_ARG, "sgmc_glm_check_table: chain %d has a null pointer", c);
    SGMC_REQUIRE(ch.D >= 1 && ch.D <= kMaxD && ch.dclass == dclass_of(ch.D), SGMC_E_ARG,
                 "sgmc_glm_check_table: chain %d: D=%d or dclass %d", c, ch.D, ch.dclass);
    SGMC_REQUIRE(ch.n >= 1 && ch.N >= 1 && ch.N <= 2147483647LL, SGMC_E_ARG,
                 "sgmc_glm_check_table: chain %d: n=%d, N=%lld", c, ch.n, (long long)ch.N);
    SGMC_REQUIRE(ch.ldx % 4 == 0 && ch.ldx >= 4 * ((ch.D + 3) / 4) &&
                     ((uintptr_t)ch.X & 15) == 0,
                 SGMC_E_ARG, "sgmc_glm_check_table: chain %d: rows not 16-byte aligned", c);
    SGMC_REQUIRE(ch.nblocks >= 1 && ch.block_begin >= 0 &&
                     (int64_t)ch.block_begin + ch.nblocks <= nblocks,
                 SGMC_E_ARG, "sgmc_glm_check_table: chain %d: blocks [%d, %d) outside the grid",
                 c, ch.block_begin, ch.block_begin + ch.nblocks);
    // a block stages the likelihoods of its ceil(n / nblocks) rows in LDS
    SGMC_REQUIRE((ch.n + ch.nblocks - 1) / ch.nblocks <= kLdsRows, SGMC_E_ARG,
                 "sgmc_glm_check_table: chain %d: %d rows over %d blocks exceed %d rows per "
                 "block", c, ch.n, ch.nblocks, kLdsRows);
    if (loop) {
      // the loop launch runs chain c on block c (block_begin is not read)
      SGMC_REQUIRE(ch.nblocks == 1, SGMC_E_ARG,
                   "sgmc_glm_check_table: chain %d has %d blocks; a loop launch needs one", c,
                   ch.nblocks);
    } else if (!block_chain) {
      SGMC_REQUIRE(ch.nblocks == per && ch.block_begin == c * per, SGMC_E_ARG,
                   "sgmc_glm_check_table: chain %d must own blocks [%d, %d)", c, c * per,
                   (c + 1) * per);
    } else {
      for (int b = ch.block_begin; b < ch.block_begin + ch.nblocks; ++b)
        SGMC_REQUIRE(block_chain[b] == c, SGMC_E_ARG,
                     "sgmc_glm_check_table: block %d maps to chain %d, not %d", b,
                     block_chain[b], c);
    }
    covered += ch.nblocks;
  }
  // Every chain's range maps to it and the ranges add up to the grid: the ranges tile
  // the grid and every map entry names its owner.
  SGMC_REQUIRE(covered == nblocks, SGMC_E_ARG,
               "sgmc_glm_check_table: chains own %lld of %d blocks", (long long)covered, nblocks);
  return SGMC_OK;
}

int sgmc_glm_fused_step(const sgmc_glm_chain* chains, int nchains, const int32_t* block_chain,
                        int nblocks, int uniform_dclass, int family, float sigma, int has_prior,
                        float prior_scale, float pot_temperature, int mode, int step, int steps,
                        float friction, float alpha, float lmbd, const float* inv_mass,
                        const float* sqrt_mass, const float* eps_table, int table_len,
                        const int32_t* save_slot, int32_t* iter, unsigned* done,
                        int advance_iter, void* stream) {
  sgmc_glm_run r = {};
  r.chains = chains;
  r.block_chain = block_chain;
  r.inv_mass = inv_mass;
  r.sqrt_mass = sqrt_mass;
  r.eps_table = eps_table;
  r.save_slot = save_slot;
  r.iter = iter;
  r.done = done;
  r.stream = stream;
  r.nchains = nchains;
  r.nblocks = nblocks;
  r.uniform_dclass = uniform_dclass;
  r.family = family;
  r.has_prior = has_prior;
  r.mode = mode;
  r.steps = steps;
  r.table_len = table_len;
  r.sigma = sigma;
  r.prior_scale = prior_scale;
  r.pot_temperature = pot_temperature;
  r.friction = friction;
  r.alpha = alpha;
  r.lmbd = lmbd;
  const int rc = check_run("sgmc_glm_fused_step", r);
  if (rc != SGMC_OK) return rc;
  const int launches = std::max(steps, launches_of(r));  // SGLD: any of the caller's steps
  SGMC_REQUIRE(step >= 0 && step < launches, SGMC_E_ARG,
               "sgmc_glm_fused_step: launch %d of %d", step, launches);
  FusedArgs a = run_args(r);
  a.step = step;
  a.advance = advance_iter ? 1 : 0;
  launch_step(r, a);
  return check_launch("sgmc_glm_fused_step");
}

int sgmc_glm_fused_run(const sgmc_glm_run* runs, int nruns) {
  SGMC_REQUIRE(runs && nruns >= 1, SGMC_E_ARG, "sgmc_glm_fused_run: no tables");
  for (int k = 0; k < nruns; ++k) {
    const sgmc_glm_run& r = runs[k];
    const int rc = check_run("sgmc_glm_fused_run", r);
    if (rc != SGMC_OK) return rc;
    SGMC_REQUIRE(r.nops >= 0 && (r.ops || r.nops == 0), SGMC_E_ARG,
                 "sgmc_glm_fused_run: no operations");
    for (int i = 0; i < r.nops; ++i) {
      const int op = r.ops[2 * i];
      SGMC_REQUIRE(op >= SGMC_OP_ITERATIONS && op <= SGMC_OP_SWAP && r.ops[2 * i + 1] >= 0,
                   SGMC_E_ARG, "sgmc_glm_fused_run: operation (%d, %d)", op, r.ops[2 * i + 1]);
      SGMC_REQUIRE(op != SGMC_OP_LOOP || (loop_mode(r.mode) && r.nblocks == r.nchains),
                   SGMC_E_ARG, "sgmc_glm_fused_run: a loop launch of mode %d, %d blocks for %d "
                   "chains", r.mode, r.nblocks, r.nchains);
      SGMC_REQUIRE(op != SGMC_OP_SWAP || (r.pairs && r.npairs >= 1 && r.nchains >= 2 &&
                                          r.swap_every >= 1),
                   SGMC_E_ARG, "sgmc_glm_fused_run: a swap launch without pairs");
    }
  }
  // (the entry points allocate nothing: more tables go in groups of kTogether)
  for (int k = 0; k < nruns; k += kTogether) {
    const int rc = issue_runs(runs + k, std::min(kTogether, nruns - k));
    if (rc != SGMC_OK) return rc;
  }
  return SGMC_OK;
}

int sgmc_glm_fused_loop(const sgmc_glm_chain* chains, int nchains, int uniform_dclass,
                        int family, float sigma, int has_prior, float prior_scale,
                        float pot_temperature, int mode, int steps, float friction, float alpha,
                        float lmbd, const float* inv_mass, const float* sqrt_mass,
                        const float* eps_table, int table_len, const int32_t* save_slot,
                        int32_t* iter, unsigned* done, int iterations, void* stream) {
  SGMC_REQUIRE(chains && eps_table && iter && done, SGMC_E_ARG,
               "sgmc_glm_fused_loop: null pointer");
  SGMC_REQUIRE(nchains >= 1 && table_len >= 1 && iterations >= 0, SGMC_E_ARG,
               "sgmc_glm_fused_loop: bad sizes");
  SGMC_REQUIRE(family == SGMC_LIK_LINEAR_GAUSSIAN || family == SGMC_LIK_LOGISTIC, SGMC_E_ARG,
               "sgmc_glm_fused_loop: unknown family %d", family);
  SGMC_REQUIRE(loop_mode(mode), SGMC_E_ARG, "sgmc_glm_fused_loop: mode %d needs a test between iterations",
               mode);
  SGMC_REQUIRE(steps >= 1, SGMC_E_ARG, "sgmc_glm_fused_loop: steps %d", steps);
  SGMC_REQUIRE(pot_temperature != 0.0f, SGMC_E_ARG, "sgmc_glm_fused_loop: temperature is zero");
  if (iterations == 0) return SGMC_OK;
  sgmc_glm_run r = {};
  r.chains = chains;
  r.inv_mass = inv_mass;
  r.sqrt_mass = sqrt_mass;
  r.eps_table = eps_table;
  r.save_slot = save_slot;
  r.iter = iter;
  r.done = done;
  r.stream = stream;
  r.nchains = r.nblocks = nchains;
  r.uniform_dclass = uniform_dclass;
  r.family = family;
  r.has_prior = has_prior;
  r.mode = mode;
  r.steps = steps;
  r.table_len = table_len;
  r.sigma = sigma;
  r.prior_scale = prior_scale;
  r.pot_temperature = pot_temperature;
  r.friction = friction;
  r.alpha = alpha;
  r.lmbd = lmbd;
  FusedArgs a = run_args(r);
  a.advance = -1;
  launch_loop_mode(r, iterations, a);
  return check_launch("sgmc_glm_fused_loop");
}

}  // extern "C"
