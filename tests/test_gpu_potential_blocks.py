"""Block splits of the minibatch potential and the row gather at their edges (GPU):
one- and two-level reductions around 32 blocks and around one run of 16 blocks more or less,
a workspace with room for one counter, one that is not 8-byte aligned, blocks without rows;
gathers of 1-, 4- and 16-byte elements around one element per thread, with indices outside
the source. Potentials: 1e-5 relative to the float64 oracle, as for every potential."""
import numpy as np
import pytest
import torch

from oracle import model as om

from jax_sgmc_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("blocks,D,floats,shift", [
    (1, 33, "all", 0), (32, 100, "all", 0), (33, 100, "all", 0), (47, 129, "all", 0),
    (48, 7, "all", 0), (49, 7, "all", 0), (1100, 65, "all", 0), (49, 301, "one counter", 0),
    (40, 96, "all", 1), (31, 1024, "all", 1)])
def test_potential_block_splits(blocks, D, floats, shift):
  print(blocks, D, floats, shift, flush=True)
  n, N = 1100 if blocks > 700 else 700, 3000
  rng = np.random.default_rng(blocks + D)
  X = (rng.standard_normal((n, D)) / np.sqrt(D)).astype(np.float32)
  y = (rng.random(n) < 0.5).astype(np.float32)
  w = (0.3 * rng.standard_normal(D)).astype(np.float32)
  ld = (D + 3) // 4 * 4
  Xp = np.zeros((n, ld), np.float32)
  Xp[:, :D] = X
  Xd, yd, wd = (torch.as_tensor(v, device=DEV) for v in (Xp, y, w))
  records = blocks * (ld + 2)
  size = int(L.query("sgmc_glm_workspace_floats", n, D, blocks)) if floats == "all" else records + 4
  ws = torch.zeros(size + shift, device=DEV)[shift:]
  U, g, var = torch.empty(1, device=DEV), torch.empty(D, device=DEV), torch.empty(1, device=DEV)
  fam = om.Family("logistic", X, y)
  Ur, gr, lik = om.stochastic_potential(fam, w, np.arange(n), 1.0, 1.0)
  scale = N / n  # the oracle's family has n rows; the call's data set N
  lp, dlp = om.gaussian_logprior(w, 1.0)
  Ur, gr = scale * (Ur + lp) - lp, scale * (gr + dlp) - dlp
  outs = []
  for _ in range(3):  # the counters return to zero
    L.call("sgmc_glm_potential", L.LIK_LOGISTIC, L.ptr(Xd), ld, L.ptr(yd), None, n, N, D,
           L.ptr(wd), 1.0, 1, 1.0, 1.0, L.ptr(U), L.ptr(g), None, L.ptr(var), L.ptr(ws),
           ws.numel(), blocks, L.stream())
    outs.append(torch.cat([U, g, var]).clone())
  assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
  got = outs[0].cpu().double().numpy()
  assert abs(got[0] - Ur) <= 1e-5 * abs(Ur)
  assert np.all(np.abs(got[1:-1] - gr) <= 1e-5 * np.abs(gr) + 1e-5 * np.max(np.abs(gr)))
  assert abs(got[-1] - np.var(lik)) <= 1e-4 * np.var(lik)


@pytest.mark.parametrize("dtype,row,rows", [
    (torch.uint8, 1, 700), (torch.uint8, 7, 255), (torch.int32, 1, 1), (torch.int32, 3, 700),
    (torch.float32, 4, 257), (torch.float32, 304, 1725), (torch.float32, 304, 6900),
    (torch.float32, 1, 524288), (torch.float32, 1, 524289), (torch.float32, 5, 131072)])
def test_gather_rows(dtype, row, rows):
  print(dtype, row, rows, flush=True)
  g = torch.Generator(device=DEV).manual_seed(row + rows)
  src = torch.randint(0, 250, (1000, row), generator=g, device=DEV).to(dtype)
  idx = torch.randint(0, 1000, (rows,), generator=g, device=DEV, dtype=torch.int32)
  if rows > 2:
    idx[1], idx[rows - 1] = -1, 1000
  want = torch.full((rows, row), 77, device=DEV).to(dtype)
  ok = (idx >= 0) & (idx < 1000)
  want[ok] = src[idx[ok].long()]
  out = torch.full((rows, row), 77, device=DEV).to(dtype)
  es = src.element_size()
  L.call("sgmc_gather_rows", L.ptr(src), 1000, L.ptr(idx), L.ptr(out), rows, row * es, row * es,
         L.stream())
  assert torch.equal(out, want)


@pytest.mark.parametrize("N,D,rows", [
    (1, 1, 1), (3, 5, 128), (257, 17, 64), (1000, 64, 63), (1000, 96, 1000), (1003, 128, 100),
    (2047, 129, 2048), (1500, 257, 129), (900, 511, 128), (700, 1000, 77), (530, 1024, 265)])
@pytest.mark.parametrize("family", ["linear_gaussian", "logistic"])
def test_full_potential_splits(N, D, rows, family):
  """Blocks and wavefronts with fewer rows than a row group, with none, and row lengths at
  the edges of the row classes: 1e-6 relative to the float64 oracle."""
  print(family, N, D, rows, flush=True)
  rng = np.random.default_rng(N + D)
  X = (rng.standard_normal((N, D)) / np.sqrt(D)).astype(np.float32)
  y = (rng.random(N) < 0.5).astype(np.float32)
  w = (0.3 * rng.standard_normal(D)).astype(np.float32)
  ld = (D + 3) // 4 * 4
  Xp = np.full((N, ld), 9.0, np.float32)  # the padding is not read into the sums
  Xp[:, :D] = X
  Xd, yd, wd = (torch.as_tensor(v, device=DEV) for v in (Xp, y, w))
  ws = torch.zeros(int(L.query("sgmc_glm_full_workspace_doubles", N, rows)), device=DEV,
                   dtype=torch.float64)
  out = torch.empty((), dtype=torch.float64, device=DEV)
  fam = L.LIK_LOGISTIC if family == "logistic" else L.LIK_LINEAR_GAUSSIAN
  for _ in range(2):
    L.call("sgmc_glm_full_potential", fam, L.ptr(Xd), ld, L.ptr(yd), N, D, L.ptr(wd), 0.7, 1, 2.0,
           1.5, L.ptr(out), L.ptr(ws), ws.numel(), rows, L.stream())
    lik, _ = (om.logistic(w, X, y) if family == "logistic" else om.linear_gaussian(w, X, y, 0.7))
    want = (-np.sum(lik) - om.gaussian_logprior(w, 2.0)[0]) / 1.5
    assert abs(out.item() - want) <= 1e-6 * abs(want)


@pytest.mark.parametrize("N,D,C", [
    (1, 1, 1), (31, 16, 3), (33, 17, 33), (700, 64, 64), (701, 65, 32), (1000, 90, 20),
    (1023, 128, 40), (1000, 129, 7), (999, 256, 64), (650, 257, 33), (640, 300, 64),
    (1300, 511, 65), (900, 512, 64), (777, 513, 20), (500, 1000, 70), (320, 1024, 33)])
def test_full_potential_of_chains_splits(N, D, C):
  """The split-fp16 full potential at the edges of its column shares (64, 128, 256, 512
  columns over 1, 2, 4 and 8 wavefronts), chain tiles and row tiles, with blocks without rows:
  2e-6 relative to float64 (1e-6 per row dot product). Padding beyond D holds large values."""
  print(N, D, C, flush=True)
  rng = np.random.default_rng(N + D + C)
  X = (rng.standard_normal((N, D)) / np.sqrt(D)).astype(np.float32)
  y = (rng.random(N) < 0.5).astype(np.float32)
  ld = (D + 3) // 4 * 4 + 4
  Xp = np.full((N, ld), 5.0, np.float32)
  Xp[:, :D] = X
  th = (0.5 * rng.standard_normal((C, D))).astype(np.float32)
  Xd, yd = torch.as_tensor(Xp, device=DEV), torch.as_tensor(y, device=DEV)
  thd = torch.as_tensor(th, device=DEV)
  exp = 14 - int(np.frexp(np.abs(X).max())[1])
  nb = 37
  ws = torch.zeros(int(L.query("sgmc_glm_full_chains_workspace_doubles", nb)), device=DEV,
                   dtype=torch.float64)
  out = torch.empty(C, dtype=torch.float64, device=DEV)
  z = X.astype(np.float64) @ th.astype(np.float64).T
  for fam, lik in ((L.LIK_LOGISTIC, y[:, None] * z - np.logaddexp(0, z)),
                   (L.LIK_LINEAR_GAUSSIAN,
                    (np.log(2 * np.pi * 0.49) + (y[:, None] - z) ** 2 / 0.49) / -2.0)):
    L.call("sgmc_glm_full_potential_chains_split", fam, L.ptr(Xd), ld, L.ptr(yd), N, D, L.ptr(thd),
           D, C, 0.7, 1, 2.0, 1.5, exp, L.ptr(out), L.ptr(ws), ws.numel(), nb, L.stream())
    got = out.cpu().numpy()
    for c in range(C):
      want = (-np.sum(lik[:, c]) - om.gaussian_logprior(th[c], 2.0)[0]) / 1.5
      assert abs(got[c] - want) <= 2e-6 * abs(want), (fam, c, got[c], want)
