"""The work that programs built on this framework have it do, as cases for timing.

Each case names a path through the public entry points with its sizes:

  grad     one minibatch gradient as a program with a loop of its own takes it:
           DeviceNumpyDataLoader.get_random_data, then value_and_grad of a GLM potential
  full     the full-data potential of one GLM chain (potential.full_potential)
  alias    a whole call of alias.sgld, from the initial sample to numpy arrays
  glm      iterations of a chain table (fused.FusedGLM, or two tables from 16 chains of
           several blocks on, as the aliases build them): SGLD, rms_prop, SGHMC, OBABO
  mh       the same with AMAGOLD's or SGGMC's full-data Metropolis-Hastings test
  ladder   reSGLD tempering ladders, a table per row length, a swap round at the end
  mlpgrad  forward and backward of mlp.MLPPotential
  mlp      iterations of mlp.FusedMLP: SGLD (plain, rms_prop), OBABO, SGGMC

``prepare`` holds what such a program keeps (dataset on the device, engine, keys), ``run``
is one pass and returns the state it computes, ``exact`` gives the same values in float64
from plain torch, random numbers (jax's Threefry-2x32 derivation) included.
"""
import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import alias, data, fused, likelihoods, mlp, potential  # noqa: E402

DEV = "cuda"
MASK = 0xFFFFFFFF
SWAP_EVERY = 50
TABLE = 256  # entries of the step-size tables


def listed():
  return [
      # a small Bayesian linear regression stepped by a user's own loop: latency of three
      # launches and the host path around them
      dict(name="grad-linreg-small", kind="grad", family="linear_gaussian", N=10_000, D=32,
           n=128),
      # a large, odd minibatch of a logistic regression (variance reduction, MAP fits)
      dict(name="grad-logistic-large", kind="grad", family="logistic", N=400_003, D=301,
           n=40_001),
      # the MH test of a generic single chain, model comparison: one pass over the data
      dict(name="full-logistic", kind="full", family="logistic", N=1_000_000, D=512),
      # quickstart-sized SGLD linear regression, the whole call
      dict(name="alias-sgld-linreg", kind="alias", family="linear_gaussian", N=10_000, D=32,
           n=128, iterations=1000),
      # preconditioned SGLD of a mid-size logistic regression with an unpadded row length
      dict(name="psgld-logistic-c16", kind="glm", family="logistic", mode="sgld_rms", C=16,
           N=200_003, D=100, n=1000, steps=1, iterations=20),
      # SGHMC on the benchmark's logistic regression, 64 chains
      dict(name="sghmc-logistic-c64", kind="glm", family="logistic", mode="sghmc", C=64,
           N=1_000_000, D=512, n=4096, steps=5, iterations=2),
      # tempering ladders over problems of mixed sizes, one swap round
      dict(name="resgld-ladders-32x8", kind="ladder", problems=32, rungs=8, n=512,
           Nmin=2_000, Nmax=200_000),
      # AMAGOLD on the benchmark's data: reversible leapfrog and a full-data test
      dict(name="amagold-logistic-c64", kind="mh", family="logistic", mode="amagold", C=64,
           N=1_000_000, D=512, n=4096, steps=5, iterations=1),
      # SGGMC of a linear regression, few chains and odd sizes
      dict(name="sggmc-linreg-c20", kind="mh", family="linear_gaussian", mode="sggmc", C=20,
           N=300_007, D=90, n=2000, steps=10, iterations=1),
      # potential and gradient of the MLP classifier as a torch autograd value, float32
      # (the aliases' default precision)
      dict(name="mlp-grad-fp32-c4", kind="mlpgrad", precision="fp32", C=4, N=20_000, D=3072,
           H1=512, H2=512, n=256),
      # preconditioned SGLD of the MLP classifier, bf16 GEMMs, 16 chains
      dict(name="psgld-mlp-bf16-c16", kind="mlp", precision="bf16", integrator="sgld", rms=True,
           C=16, N=50_000, D=3072, H1=512, H2=512, n=256, steps=1, iterations=2),
      # SGGMC of the wider MLP classifier, e4m3 GEMMs: proposals of the alias's default
      # ten OBABO steps, the full potential over all rows and the test
      dict(name="sggmc-mlp-fp8-c16", kind="mlp", precision="fp8", integrator="sggmc", rms=False,
           C=16, N=50_000, D=3072, H1=1024, H2=1024, n=512, steps=10, iterations=1),
  ]


def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(["grad", "full", "alias", "glm", "glm", "glm", "mh", "mh", "ladder",
                     "mlpgrad", "mlp", "mlp"])
  family = rng.choice(["linear_gaussian", "logistic"])
  D = _log_int(rng, 3, 1024)
  N = min(_log_int(rng, 5_000, 1_000_000), 400_000_000 // D)
  if kind == "grad":
    return dict(kind=kind, family=family, N=N, D=D, n=min(N, _log_int(rng, 32, 60_000)))
  if kind == "full":
    return dict(kind=kind, family=family, N=N, D=D)
  if kind == "alias":
    return dict(kind=kind, family=family, N=N, D=min(D, 256), n=min(N, _log_int(rng, 16, 1000)),
                iterations=_log_int(rng, 100, 1000))
  if kind == "glm":
    return dict(kind=kind, family=family,
                mode=rng.choice(["sgld", "sgld_rms", "sghmc", "obabo"]), C=_log_int(rng, 1, 64),
                N=N, D=D, n=min(N, _log_int(rng, 32, 4096)), steps=rng.randint(1, 10),
                iterations=rng.randint(1, 5))
  if kind == "mh":
    return dict(kind=kind, family=family, mode=rng.choice(["amagold", "sggmc"]),
                C=_log_int(rng, 2, 64), N=N, D=D, n=min(N, _log_int(rng, 64, 4096)),
                steps=rng.randint(1, 10), iterations=rng.randint(1, 2))
  if kind == "ladder":
    return dict(kind=kind, problems=rng.randint(4, 32), rungs=rng.randint(2, 8),
                n=_log_int(rng, 64, 512), Nmin=2_000, Nmax=_log_int(rng, 10_000, 200_000))
  dims = dict(D=64 * _log_int(rng, 2, 48), H1=128 * rng.randint(1, 8), H2=128 * rng.randint(1, 8),
              n=64 * rng.randint(1, 8))
  if kind == "mlpgrad":
    return dict(kind=kind, precision=rng.choice(["fp32", "bf16", "fp8"]), C=rng.randint(1, 8),
                N=_log_int(rng, 2_000, 50_000), **dims)
  integrator = rng.choice(["sgld", "obabo", "sggmc"])
  return dict(kind=kind, precision=rng.choice(["fp32", "bf16", "fp8"]), integrator=integrator,
              rms=integrator == "sgld" and rng.random() < 0.5, C=rng.randint(1, 8),
              N=_log_int(rng, 2_000, 50_000), steps=1 if integrator == "sgld" else rng.randint(1, 4),
              iterations=rng.randint(1, 2), **dims)


# ------------------------------------------------------------------ inputs ----

def _gen(seed):
  return torch.Generator(device=DEV).manual_seed(seed)


def _words(seed, count):
  """``count`` jax keys (two uint32 words each)."""
  return np.random.default_rng(seed).integers(0, 2 ** 32, size=(count, 2), dtype=np.uint32)


def _align4(x):
  return (x + 3) // 4 * 4


def _glm_data(family, N, D, g):
  """Rows N(0, 1) / sqrt(D) padded to a multiple of four floats, true weights N(0, 1),
  responses with noise 0.5 or Bernoulli labels."""
  X = torch.zeros((N, _align4(D)), device=DEV)
  X[:, :D].copy_(torch.randn((N, D), generator=g, device=DEV).mul_(1.0 / math.sqrt(D)))
  w = torch.randn(D, generator=g, device=DEV)
  z = X[:, :D] @ w
  if family == "logistic":
    y = (torch.rand(N, generator=g, device=DEV) < torch.sigmoid(z)).to(torch.float32)
  else:
    y = z + 0.5 * torch.randn(N, generator=g, device=DEV)
  return X, y, w


def _likelihood(family):
  return likelihoods.Logistic() if family == "logistic" else likelihoods.LinearGaussian(0.5)


def _glm_inputs(case, seed):
  g = _gen(seed)
  X, y, w = _glm_data(case["family"], case["N"], case["D"], g)
  C = case.get("C", 1)
  theta0 = w[None] + 0.1 * torch.randn((C, case["D"]), generator=g, device=DEV)
  return X, y, theta0


def _glm_eps(case):
  """Stable step sizes: a unit of curvature per row over D columns, N rows, unit prior."""
  curv = case["N"] / case["D"] * (4.0 if case["family"] == "linear_gaussian" else 0.25) + 1.0
  if case.get("mode") in ("sgld_rms",):
    first = 1e-3
  elif case.get("mode") in (None, "sgld"):
    first = 0.1 / curv
  elif case["kind"] == "mh":
    first = 0.005 / math.sqrt(curv)  # small enough that proposals are accepted and rejected
  else:
    first = 0.1 / math.sqrt(curv)
  k = np.arange(TABLE, dtype=np.float32)
  return (np.float32(first) * (1.0 + 0.01 * k) ** np.float32(-0.33)).astype(np.float32)


def _ladder_inputs(case, seed):
  """Problems of row lengths cycling 16, 64, 256, 1024, log-uniform row counts."""
  g = _gen(seed)
  rng = np.random.default_rng(seed)
  probs = []
  for k in range(case["problems"]):
    D = (16, 64, 256, 1024)[k % 4]
    N = int(round(math.exp(rng.uniform(math.log(case["Nmin"]), math.log(case["Nmax"])))))
    X, y, _ = _glm_data("logistic", N, D, g)
    probs.append((X, y))
  C = case["problems"] * case["rungs"]
  temps = [20.0 ** (j / max(1, case["rungs"] - 1)) for j in range(case["rungs"])]
  words = _words(seed, 3 * C)
  return probs, temps, words[:C], words[C:2 * C], words[2 * C:]


def _ladder_eps():
  k = np.arange(1000, dtype=np.float32)
  return (np.float32(1e-3) * (1.0 + 0.01 * k) ** np.float32(-0.33)).astype(np.float32)


def _mlp_inputs(case, seed):
  g = _gen(seed)
  D, H1, H2, C, N = case["D"], case["H1"], case["H2"], case["C"], case["N"]
  X = torch.rand((N, D), generator=g, device=DEV)
  labels = torch.argmax((X - 0.5) @ torch.randn((D, mlp.NCLS), generator=g, device=DEV),
                        dim=1).to(torch.int32)
  theta0 = torch.zeros((C, mlp.param_count(D, H1, H2)), device=DEV)
  off = 0
  for rows, cols in ((D, H1), (H1, H2), (H2, mlp.NCLS)):
    theta0[:, off:off + rows * cols] = math.sqrt(2.0 / rows) * torch.randn(
        (C, rows * cols), generator=g, device=DEV)
    off += rows * cols
  return X, labels, theta0


def _mlp_eps(case):
  return np.full(TABLE, 1e-5 if case["integrator"] == "sgld" else 1e-4, np.float32)


# ----------------------------------------------------------------- prepare ----

def prepare(case, seed):
  return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"], case=case)


def _prepare_grad(case, seed):
  X, y, theta0 = _glm_inputs(case, seed)
  loader = data.DeviceNumpyDataLoader(x=X[:, :case["D"]], y=y)
  pot = potential.minibatch_potential(likelihoods.GaussianPrior(1.0), _likelihood(case["family"]))
  key = torch.as_tensor(_words(seed, 1)[0].view(np.int32).copy(), device=DEV)
  return dict(loader=loader, pot=pot, w=theta0[0].clone(), key=key)


def _prepare_full(case, seed):
  X, y, theta0 = _glm_inputs(case, seed)
  loader = data.DeviceNumpyDataLoader(x=X[:, :case["D"]], y=y)
  pot = potential.full_potential(likelihoods.GaussianPrior(1.0), _likelihood(case["family"]))
  init, full_map, _ = data.full_reference_data(loader, min(1024, case["N"]))
  return dict(pot=pot, w=theta0[0].clone(), data_state=init(), full_map=full_map)


def _alias_steps(case):
  first = float(_glm_eps(case)[0])
  return first, 0.1 * first


def _prepare_alias(case, seed):
  X, y, theta0 = _glm_inputs(case, seed)
  loader = data.DeviceNumpyDataLoader(x=X[:, :case["D"]], y=y)
  pot = potential.minibatch_potential(likelihoods.GaussianPrior(1.0), _likelihood(case["family"]))
  first, last = _alias_steps(case)
  run_fn = alias.sgld(pot, loader, cache_size=1, batch_size=case["n"], first_step_size=first,
                      last_step_size=last, burn_in=case["iterations"] // 2,
                      accepted_samples=None)
  words = _words(seed, 2)
  return dict(run_fn=run_fn, sample=theta0[0].clone(), key=words[0], dkey=words[1])


def _chains(case, seed):
  X, y, theta0 = _glm_inputs(case, seed)
  words = _words(seed, 2 * case["C"])
  th = theta0.cpu().numpy()
  return [dict(X=X, y=y, D=case["D"], n=case["n"], theta0=th[c], key=tuple(words[c]),
               dkey=tuple(words[case["C"] + c])) for c in range(case["C"])], words


def _glm_kwargs(case):
  return dict(steps=case["steps"], friction=0.5, sigma=0.5, prior_scale=1.0)


def _prepare_glm(case, seed):
  chains, _ = _chains(case, seed)
  args = (case["family"], case["mode"], _glm_eps(case))
  total = case["C"] * case["n"] * 4 * _align4(case["D"])
  multi = fused.blocks_for(case["n"], case["D"], max(64 * 1024, total // 2048)) > 1
  if case["C"] >= 16 and multi:
    eng = fused.TableGroup.split(chains, 2, *args, **_glm_kwargs(case))
    return dict(eng=eng, tables=eng.engines)
  eng = fused.FusedGLM(chains, *args, **_glm_kwargs(case))
  return dict(eng=eng, tables=[eng])


def _prepare_mh(case, seed):
  chains, words = _chains(case, seed)
  eng = fused.FusedGLM(chains, case["family"], case["mode"], _glm_eps(case), **_glm_kwargs(case))
  test = fused.AmagoldMH if case["mode"] == "amagold" else fused.SggmcMH
  return dict(eng=eng, tables=[eng],
              mh=test(eng, keys=[tuple(words[c]) for c in range(case["C"])]))


def _prepare_ladder(case, seed):
  probs, temps, keys, dkeys, skeys = _ladder_inputs(case, seed)
  R = case["rungs"]
  tables = []
  for D in (16, 64, 256, 1024):
    chains, pairs, ptemps, parity, sk = [], [], [], [], []
    for k, (X, y) in enumerate(probs):
      if X.shape[1] != D:
        continue
      for j in range(R):
        c = k * R + j
        chains.append(dict(X=X, y=y, D=D, n=case["n"], theta0=np.zeros(D, np.float32),
                           key=tuple(keys[c]), dkey=tuple(dkeys[c]), temperature=temps[j],
                           save=False))
        if j + 1 < R:
          pairs.append((len(chains) - 1, len(chains)))
          ptemps.append((temps[j], temps[j + 1]))
          parity.append(j % 2)
          sk.append(tuple(skeys[c]))
    eng = fused.FusedGLM(chains, "logistic", "sgld", _ladder_eps(), prior_scale=1.0,
                         target_bytes=(1 << 30) if D <= 64 else None)
    fused.ReplicaExchange(eng, pairs, ptemps, keys=sk, swap_every=SWAP_EVERY, parity=parity)
    tables.append(eng)
  return dict(eng=fused.TableGroup(tables, stream_of=[0, 0, 1, 2]), tables=tables)


def _mlp_engine(case, seed, **kw):
  X, labels, theta0 = _mlp_inputs(case, seed)
  words = _words(seed, 2 * case["C"])
  eng = mlp.FusedMLP(X, labels, (case["D"], case["H1"], case["H2"]), case["n"],
                     theta0.cpu().numpy(), keys=words[:case["C"]], dkeys=words[case["C"]:],
                     prior_scale=1.0, precision=case["precision"], **kw)
  return eng, theta0


def _prepare_mlpgrad(case, seed):
  eng, theta0 = _mlp_engine(case, seed, eps_table=np.full(1, 1e-5, np.float32))
  return dict(eng=eng, theta=theta0.clone().requires_grad_(True))


def _prepare_mlp(case, seed):
  eng, _ = _mlp_engine(case, seed, eps_table=_mlp_eps(case), rms=case["rms"],
                       integrator=case["integrator"], friction=0.5, steps=case["steps"])
  return dict(eng=eng)


_PREPARE = dict(grad=_prepare_grad, full=_prepare_full, alias=_prepare_alias, glm=_prepare_glm,
                mh=_prepare_mh, ladder=_prepare_ladder, mlpgrad=_prepare_mlpgrad,
                mlp=_prepare_mlp)


# --------------------------------------------------------------------- run ----

def run(state):
  kind, case = state["kind"], state["case"]
  if kind == "grad":
    state["key"], batch = state["loader"].get_random_data(state["key"], case["n"])
    (U, _), grad = state["pot"].value_and_grad(state["w"], batch)
    return {"U": U, "grad": grad}
  if kind == "full":
    U, (state["data_state"], _) = state["pot"](state["w"], state["data_state"],
                                               state["full_map"])
    return {"U": U}
  if kind == "alias":
    return state["run_fn"](state["sample"], iterations=case["iterations"],
                           keys=[state["key"]], data_keys=[state["dkey"]])
  if kind == "mlpgrad":
    state["theta"].grad = None
    U = mlp.MLPPotential.apply(state["theta"], state["eng"])
    U.sum().backward()
    return {"U": U.detach(), "grad": state["theta"].grad}
  eng = state["eng"]
  if kind == "mlp":
    eng.run(case["iterations"])
    out = {"theta": eng.theta, "U": eng.U}
    if case["rms"]:
      out["v"] = eng.v
    if eng.mom is not None:
      out["mom"] = eng.mom
    if eng.U_full is not None:
      out["U_full"] = eng.U_full
    return out
  eng.run(SWAP_EVERY if kind == "ladder" else case["iterations"])
  out = {"theta": [t.theta_flat for t in state["tables"]], "U": [t.U for t in state["tables"]]}
  if state["tables"][0].mom_flat is not None:
    out["mom"] = [t.mom_flat for t in state["tables"]]
  if state["tables"][0].v_flat is not None:
    out["v"] = [t.v_flat for t in state["tables"]]
  if kind == "mh":
    out["U_full"] = state["mh"].U_full
  return out


# -------------------------------------------------------------------- work ----

def work(case):
  """Rows read once, parameters and state read and written once, per evaluation."""
  kind, D = case["kind"], case.get("D", 0)
  rows = lambda n: n * (4 * D + 4)
  if kind == "grad":
    return {"bytes": rows(case["n"]) + 8 * D, "flops": 4 * case["n"] * D}
  if kind == "full":
    return {"bytes": rows(case["N"]) + 4 * D, "flops": 2 * case["N"] * D}
  if kind == "alias":
    its = case["iterations"]
    return {"bytes": its * rows(case["n"]) + (its - its // 2) * 4 * (D + 1),
            "flops": its * 4 * case["n"] * D}
  if kind in ("glm", "mh"):
    evals = case["C"] * case["iterations"]
    if case["mode"] in ("sghmc", "amagold"):
      evals *= case["steps"]
    elif case["mode"] in ("obabo", "sggmc"):
      evals *= 2 * case["steps"]
    state = 8 * D if case["mode"] == "sgld" else 16 * D
    w = {"bytes": evals * (rows(case["n"]) + state), "flops": evals * 4 * case["n"] * D}
    if kind == "mh":
      w["bytes"] += case["iterations"] * rows(case["N"])
      w["flops"] += case["iterations"] * 2 * case["N"] * D * case["C"]
    return w
  if kind == "ladder":
    evals = SWAP_EVERY * case["rungs"]
    dims = [(16, 64, 256, 1024)[k % 4] for k in range(case["problems"])]
    return {"bytes": sum(evals * (case["n"] * (4 * d + 4) + 8 * d) for d in dims),
            "flops": sum(evals * 4 * case["n"] * d for d in dims)}
  H1, H2, C, n = case["H1"], case["H2"], case["C"], case["n"]
  P = mlp.param_count(D, H1, H2)
  macs = D * H1 + H1 * H2 + H2 * mlp.NCLS
  grad = 2 * n * (2 * macs + H1 * H2 + H2 * mlp.NCLS)
  if kind == "mlpgrad":
    return {"bytes": C * (8 * P + rows(n)), "flops": C * grad}
  evals = case["iterations"] * (1 if case["integrator"] == "sgld" else 2 * case["steps"])
  state = 16 if case["rms"] or case["integrator"] != "sgld" else 8
  w = {"bytes": C * evals * (state * P + rows(n)), "flops": C * evals * grad}
  if case["integrator"] == "sggmc":
    w["bytes"] += case["iterations"] * (rows(case["N"]) + 4 * C * P)
    w["flops"] += case["iterations"] * C * 2 * case["N"] * macs
  return w


# ------------------------------------------------------------------- exact ----
# jax's original Threefry derivation on int64 tensors; keys are [..., 2].

def _threefry(key, x0, x1):
  k0, k1 = key[..., 0:1], key[..., 1:2]
  ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA)
  x0, x1 = (x0 + ks[0]) & MASK, (x1 + ks[1]) & MASK
  for i in range(5):
    for r in ((13, 15, 26, 6), (17, 29, 16, 24))[i % 2]:
      x0 = (x0 + x1) & MASK
      x1 = (((x1 << r) | (x1 >> (32 - r))) & MASK) ^ x0
    x0 = (x0 + ks[(i + 1) % 3]) & MASK
    x1 = (x1 + ks[(i + 2) % 3] + i + 1) & MASK
  return x0, x1


def _split(key, num=2):
  j = torch.arange(num, device=key.device)
  a, b = _threefry(key, j, j + num)
  out = torch.cat([a, b], -1).reshape(key.shape[:-1] + (num, 2))
  return [out[..., i, :] for i in range(num)]


def _bits(key, S):
  m = (S + 1) // 2
  j = torch.arange(m, device=key.device)
  a, b = _threefry(key, j, torch.where(j + m < S, j + m, torch.zeros_like(j)))
  return torch.cat([a, b], -1)[..., :S]


def _unit(bits):
  return ((bits >> 9) | 0x3F800000).to(torch.int32).view(torch.float32) - 1.0


def _normal(key, S):
  lo = torch.tensor(-0.99999994, dtype=torch.float32, device=key.device)
  u = torch.maximum(lo, _unit(_bits(key, S)) * 2.0 + lo)
  return torch.erfinv(u.double()) * math.sqrt(2.0)


def _tree_normal(key, sizes):
  return torch.cat([_normal(k, s) for k, s in zip(_split(key, len(sizes)), sizes)], -1)


def _randint(key, n, N):
  k1, k2 = _split(key)
  m = 65536 % N
  mult = ((m * m) & MASK) % N
  return ((((_bits(k1, n) % N) * mult) & MASK) + _bits(k2, n) % N & MASK) % N


def _keys(words):
  return torch.as_tensor(np.asarray(words).astype(np.int64), device=DEV)


def _f32(x):
  return np.float32(x)


class _GLM:
  """Chains [G] of one dataset in float64: positions [G, D], keys [G, 2]."""

  def __init__(self, X, y, family, D, n, theta, key, dkey, temperature):
    self.X, self.y, self.family, self.D, self.n = X, y, family, D, n
    self.N = X.shape[0]
    self.theta, self.key, self.dkey = theta.double(), key, dkey
    self.T = [_f32(t) for t in temperature]
    self.p = torch.zeros_like(self.theta)
    self.v = torch.ones_like(self.theta)
    self.ke = torch.zeros((2, theta.shape[0]), dtype=torch.float64, device=DEV)

  def lik(self, z, y):
    if self.family == "logistic":
      return y * z - torch.nn.functional.softplus(z, threshold=700.0), y - torch.sigmoid(z)
    s2 = 0.25
    return (math.log(2 * math.pi * s2) + (y - z) ** 2 / s2) / -2.0, (y - z) / s2

  def log_prior(self, th):
    return ((math.log(2 * math.pi) + th * th) / -2.0).sum(-1)

  def grad(self, th):
    """U, grad U and var(lik) at th for the next minibatch of every chain."""
    self.dkey, sub = _split(self.dkey)
    idx = _randint(sub, self.n, self.N)
    x = self.X[idx][..., :self.D].double()
    lik, r = self.lik((x @ th[..., None])[..., 0], self.y[idx].double())
    g = -self.N / self.n * (r[..., None, :] @ x)[..., 0, :] + th
    return -self.N * lik.mean(-1) - self.log_prior(th), g, lik.var(-1, unbiased=False)

  def full(self, th):
    tot = torch.zeros(th.shape[0], dtype=torch.float64, device=DEV)
    for a in range(0, self.N, 65536):
      x = self.X[a:a + 65536, :self.D].double()
      tot += self.lik(x @ th.T, self.y[a:a + 65536].double()[:, None])[0].sum(0)
    return -tot - self.log_prior(th)

  def noise(self, sub):
    return _normal(_split(sub, 1)[0], self.D)

  def col(self, f):
    return torch.tensor([float(f(t)) for t in self.T], dtype=torch.float64, device=DEV)[:, None]

  def sgld(self, eps, rms=False):
    self.key, sub = _split(self.key)
    xi = self.noise(sub)
    self.U, g, self.var = self.grad(self.theta)
    sn = self.col(lambda t: np.sqrt(_f32(_f32(2) * t) * eps)) * xi
    if rms:
      self.v = 0.9 * self.v + 0.1 * g * g
      G = 1.0 / (1e-5 + torch.sqrt(self.v))
      self.theta = self.theta - float(eps) * G * g + torch.sqrt(G) * sn
    else:
      self.theta = self.theta - float(eps) * g + sn

  def sghmc(self, eps, steps, friction=0.5):
    self.key, sub = _split(self.key)
    self.p = self.noise(sub)
    for _ in range(steps):
      self.theta = self.theta + float(eps) * self.p
      self.p = self.p * (1.0 - float(_f32(eps * _f32(friction))))
      self.U, g, _ = self.grad(self.theta)
      self.key, sub = _split(self.key)
      self.p = self.p - float(eps) * g + friction * float(np.sqrt(_f32(2) * eps)) * self.noise(sub)

  def obabo(self, eps, steps, friction=0.5):
    perm = np.exp(_f32(_f32(-friction) * eps))
    decay = float(np.sqrt(perm))
    amp = self.col(lambda t: np.sqrt(_f32((_f32(1) - perm) * t)))
    half = float(_f32(0.5) * eps)
    for _ in range(steps):
      self.key, s1, s2 = _split(self.key, 3)
      p = decay * self.p + amp * self.noise(s1)
      self.ke[0] += 0.5 * (p * p).sum(-1)
      U0, g, _ = self.grad(self.theta)
      p = p - half * g
      self.theta = self.theta + float(eps) * p
      U1, g, _ = self.grad(self.theta)
      p = p - half * g
      self.ke[1] += 0.5 * (p * p).sum(-1)
      self.p = decay * p + amp * self.noise(s2)
      self.U = 0.5 * (U0 + U1)

  def amagold(self, eps, steps, friction=0.5):
    half, e = float(_f32(0.5) * eps), float(eps)
    ef = _f32(eps * _f32(friction))
    decay, rescale = float(_f32(1) - ef), float(_f32(1) / _f32(_f32(1) + ef))
    amp = float(np.sqrt(_f32(_f32(4 * friction) * eps)))
    energy = torch.zeros(self.theta.shape[0], dtype=torch.float64, device=DEV)
    for k in range(steps):
      self.theta = self.theta + (e if k else half) * self.p
      self.key, sub = _split(self.key)
      self.U, g, _ = self.grad(self.theta)
      p = rescale * (decay * self.p - e * g + amp * self.noise(sub))
      energy += half * ((self.p + p) * g).sum(-1)
      self.p = p
    self.theta = self.theta + half * self.p
    return energy

  def start_mh(self, amagold):
    self.key, self.mkey = _split(self.key)
    if amagold:
      self.key, sub = _split(self.key)
      self.p = self.noise(sub)
    self.U_full = self.full(self.theta)
    self.U = torch.zeros_like(self.U_full)

  def mh(self, case, eps):
    theta, p, U = self.theta, self.p, self.U
    self.mkey, sub = _split(self.mkey)
    log_u = torch.log(_unit(_bits(sub, 1))[:, 0].double())
    if case["mode"] == "amagold":
      energy = self.amagold(eps, case["steps"])
      new = self.full(self.theta)
      acc = log_u < torch.clamp(self.U_full - new + energy, max=0.0)
      U, p = self.U, -p
    else:
      self.ke.zero_()
      self.obabo(eps, case["steps"])
      new = self.full(self.theta)
      acc = log_u < torch.clamp(-(new - self.U_full + self.ke[1] - self.ke[0]), max=0.0)
    a = acc[:, None]
    self.theta, self.p = torch.where(a, self.theta, theta), torch.where(a, self.p, p)
    self.U_full, self.U = torch.where(acc, new, self.U_full), torch.where(acc, self.U, U)


def _glm_exact(case, seed):
  X, y, theta0 = _glm_inputs(case, seed)
  C = case["C"]
  words = _words(seed, 2 * C)
  return _GLM(X, y, case["family"], case["D"], case["n"], theta0, _keys(words[:C]),
              _keys(words[C:]), [1.0] * C)


def _flat(t):
  """[G, D] as the engines store it: rows padded with zeros to four floats."""
  return torch.nn.functional.pad(t, (0, _align4(t.shape[1]) - t.shape[1])).reshape(-1)


def _mlp_leaves(th, case):
  D, H1, H2 = case["D"], case["H1"], case["H2"]
  out, off = [], 0
  for shape in ((D, H1), (H1, H2), (H2, mlp.NCLS), (H1,), (H2,), (mlp.NCLS,)):
    size = int(np.prod(shape))
    out.append(th[off:off + size].reshape(shape))
    off += size
  return out


def _mlp_forward(th, case, x):
  W1, W2, W3, b1, b2, b3 = _mlp_leaves(th, case)
  h1 = torch.relu(x @ W1 + b1)
  h2 = torch.relu(h1 @ W2 + b2)
  return h1, h2, torch.log_softmax(h2 @ W3 + b3, -1)


def _mlp_prior(th):
  return -0.5 * (math.log(2 * math.pi) * th.numel() + torch.dot(th, th))


def _mlp_grad(th, case, X, labels, idx):
  x, lab = X[idx].double(), labels[idx].long()
  h1, h2, lp = _mlp_forward(th, case, x)
  _, W2, W3 = _mlp_leaves(th, case)[:3]
  scale = -case["N"] / case["n"]
  U = scale * lp[torch.arange(len(idx), device=DEV), lab].sum() - _mlp_prior(th)
  dL = scale * (torch.nn.functional.one_hot(lab, mlp.NCLS).double() - lp.exp())
  d2 = (dL @ W3.T) * (h2 > 0)
  d1 = (d2 @ W2.T) * (h1 > 0)
  parts = (x.T @ d1, h1.T @ d2, h2.T @ dL, d1.sum(0), d2.sum(0), dL.sum(0))
  return U, torch.cat([q.reshape(-1) for q in parts]) + th


def _mlp_full(th, case, X, labels):
  tot = torch.zeros((), dtype=torch.float64, device=DEV)
  for a in range(0, case["N"], 8192):
    lp = _mlp_forward(th, case, X[a:a + 8192].double())[2]
    tot += lp.gather(1, labels[a:a + 8192].long()[:, None]).sum()
  return -tot - _mlp_prior(th)


def _mlp_chain(case, X, labels, th, key, dkey):
  """One chain's iterations: (theta, U, v, momentum, kept full potential)."""
  sizes = [t.numel() for t in _mlp_leaves(th, case)]
  eps = _mlp_eps(case)[0]
  e, half = float(eps), float(_f32(0.5) * eps)
  v, p, U = torch.ones_like(th), torch.zeros_like(th), torch.zeros((), dtype=torch.float64,
                                                                   device=DEV)
  perm = np.exp(_f32(_f32(-0.5) * eps))
  decay, amp = float(np.sqrt(perm)), float(np.sqrt(_f32(1) - perm))
  U_full = None

  def grad():
    nonlocal dkey
    dkey, sub = _split(dkey)
    return _mlp_grad(th, case, X, labels, _randint(sub, case["n"], case["N"]))

  if case["integrator"] == "sggmc":
    key, mkey = _split(key)
    U_full = _mlp_full(th, case, X, labels)
  for _ in range(case["iterations"]):
    if case["integrator"] == "sgld":
      key, sub = _split(key)
      U, g = grad()
      sn = float(np.sqrt(_f32(2) * eps)) * _tree_normal(sub, sizes)
      if case["rms"]:
        v = 0.9 * v + 0.1 * g * g
        G = 1.0 / (1e-5 + torch.sqrt(v))
        th = th - e * G * g + torch.sqrt(G) * sn
      else:
        th = th - e * g + sn
      continue
    th0, p0, U_kept, ks, ke = th, p, U, 0.0, 0.0
    for _ in range(case["steps"]):
      key, s1, s2 = _split(key, 3)
      p = decay * p + amp * _tree_normal(s1, sizes)
      ks = ks + 0.5 * torch.dot(p, p)
      U0, g = grad()
      p = p - half * g
      th = th + e * p
      U1, g = grad()
      p = p - half * g
      ke = ke + 0.5 * torch.dot(p, p)
      p = decay * p + amp * _tree_normal(s2, sizes)
      U = 0.5 * (U0 + U1)
    if U_full is not None:
      mkey, sub = _split(mkey)
      new = _mlp_full(th, case, X, labels)
      log_u = torch.log(_unit(_bits(sub, 1))[0].double())
      if bool(log_u < torch.clamp(-(new - U_full + ke - ks), max=0.0)):
        U_full = new
      else:
        th, p, U = th0, p0, U_kept
  return th, U, v, p, U_full


def exact(case, seed):
  kind = case["kind"]
  if kind in ("grad", "full"):
    X, y, theta0 = _glm_inputs(case, seed)
    g = _GLM(X, y, case["family"], case["D"], case.get("n", 1), theta0, None,
             _keys(_words(seed, 1)), [1.0])
    if kind == "full":
      return {"U": g.full(g.theta)[0]}
    U, grad, _ = g.grad(g.theta)
    return {"U": U[0], "grad": grad[0]}
  if kind == "alias":
    X, y, theta0 = _glm_inputs(case, seed)
    words = _words(seed, 2)
    g = _GLM(X, y, case["family"], case["D"], case["n"], theta0, _keys(words[:1]),
             _keys(words[1:]), [1.0])
    # polynomial schedule a (b + i)^-0.33 between the first and last step size, float32
    its = case["iterations"]
    first, last = (_f32(s) for s in _alias_steps(case))
    gamma = _f32(0.33)
    ginv = np.power(gamma, _f32(-1.0))
    apow = _f32((np.power(last, -ginv) - np.power(first, -ginv)) / _f32(its - 1))
    a = np.power(apow, -gamma)
    b = np.power(_f32(first / a), -ginv)
    eps = (a * np.power(b + np.arange(its).astype(np.float32), -gamma)).astype(np.float32)
    th, lik = [], []
    for i in range(its):
      g.sgld(eps[i])
      if i >= its // 2:
        th.append(g.theta[0])
        lik.append(-g.U[0])
    return [{"sample_count": None, "samples": {"variables": torch.stack(th),
                                               "likelihood": torch.stack(lik)}}]
  if kind in ("glm", "mh"):
    g, eps = _glm_exact(case, seed), _glm_eps(case)
    if kind == "mh":
      g.key = _keys(_words(seed, case["C"]))
      g.start_mh(case["mode"] == "amagold")
    for i in range(case["iterations"]):
      if kind == "mh":
        g.mh(case, eps[i])
      elif case["mode"] in ("sgld", "sgld_rms"):
        g.sgld(eps[i], case["mode"] == "sgld_rms")
      else:
        getattr(g, case["mode"])(eps[i], case["steps"])
    C = case["C"]
    total = C * case["n"] * 4 * _align4(case["D"])
    multi = fused.blocks_for(case["n"], case["D"], max(64 * 1024, total // 2048)) > 1
    cut = [0, C]
    if kind == "glm" and C >= 16 and multi:
      cut = [int(c) for c in np.linspace(0, C, 3).round()]
    part = lambda t: [t[i:j] for i, j in zip(cut[:-1], cut[1:])]
    out = {"theta": [_flat(t) for t in part(g.theta)], "U": part(g.U)}
    if case["mode"] == "sgld_rms":
      # the padding of the engine's state keeps its initial ones
      out["v"] = [torch.nn.functional.pad(t, (0, _align4(t.shape[1]) - t.shape[1]),
                                          value=1.0).reshape(-1) for t in part(g.v)]
    elif case["mode"] != "sgld":
      out["mom"] = [_flat(t) for t in part(g.p)]
    if kind == "mh":
      out["U_full"] = g.U_full
    return out
  if kind == "ladder":
    return _ladder_exact(case, seed)
  X, labels, theta0 = _mlp_inputs(case, seed)
  C = case["C"]
  words = _words(seed, 2 * C)
  if kind == "mlpgrad":
    Us, gs = [], []
    for c in range(C):
      _, sub = _split(_keys(words[C + c]))
      U, g = _mlp_grad(theta0[c].double(), case, X, labels, _randint(sub, case["n"], case["N"]))
      Us.append(U)
      gs.append(g)
    return {"U": torch.stack(Us), "grad": torch.stack(gs)}
  res = [_mlp_chain(case, X, labels, theta0[c].double(), _keys(words[c]), _keys(words[C + c]))
         for c in range(C)]
  out = {"theta": torch.stack([r[0] for r in res]), "U": torch.stack([r[1] for r in res])}
  if case["rms"]:
    out["v"] = torch.stack([r[2] for r in res])
  if case["integrator"] != "sgld":
    out["mom"] = torch.stack([r[3] for r in res])
  if case["integrator"] == "sggmc":
    out["U_full"] = torch.stack([r[4] for r in res])
  return out


def _ladder_exact(case, seed):
  probs, temps, keys, dkeys, skeys = _ladder_inputs(case, seed)
  eps, R = _ladder_eps(), case["rungs"]
  by_dim = {D: [] for D in (16, 64, 256, 1024)}
  for k, (X, y) in enumerate(probs):
    D, c = X.shape[1], slice(k * R, (k + 1) * R)
    g = _GLM(X, y, "logistic", D, case["n"], torch.zeros((R, D), device=DEV), _keys(keys[c]),
             _keys(dkeys[c]), temps)
    for i in range(SWAP_EVERY):
      g.sgld(eps[i])
    for j in range(0, R - 1, 2):  # the even pairs' round
      dt = 1.0 / temps[j] - 1.0 / temps[j + 1]
      log_s = dt * ((g.U[j] - g.U[j + 1]) - dt * g.var[j])
      _, sub = _split(_keys(skeys[k * R + j]))
      if not bool(torch.log(_unit(_bits(sub, 1))[0].double()) < log_s):
        order = list(range(R))
        order[j], order[j + 1] = j + 1, j
        g.theta, g.U = g.theta[order], g.U[order]
    by_dim[D].append(g)
  return {"theta": [torch.cat([g.theta.reshape(-1) for g in gs]) for gs in by_dim.values()],
          "U": [torch.cat([g.U for g in gs]) for gs in by_dim.values()]}
