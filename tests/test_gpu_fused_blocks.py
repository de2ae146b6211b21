"""The fused GLM step at the edges of its block and row splits, against the float64 oracle
(GPU): chains of 1, 2, 16, 17 and 33 blocks (one record kept in LDS; one round of record
loads; runs of blocks summed side by side), row lengths around the 32- and 64-lane row
classes, odd lengths, minibatches that leave wavefronts without rows, and a record buffer
that is not 8-byte aligned. Bound: 1e-5 relative (floor 1e-5 max |value|), as for every fused
trajectory."""
import numpy as np
import pytest
import torch

from oracle import model as om
from oracle import steps as ost

from jax_sgmc_amd import fused
from jax_sgmc_amd import random as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
N, ITERS = 1500, 2


def _close(got, ref, what):
  got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
  tol = 1e-5 * np.abs(ref) + 1e-5 * max(1e-3, np.max(np.abs(ref)))
  assert np.all(np.abs(got - ref) <= tol), what


def _engine(D, n, mode, nb, shift):
  rng = np.random.default_rng(D + n)
  X = (rng.standard_normal((N, D)) / np.sqrt(D)).astype(np.float32)
  y = (rng.random(N) < 0.5).astype(np.float32)
  Xp = np.zeros((N, (D + 3) // 4 * 4), np.float32)
  Xp[:, :D] = X
  th0 = (0.1 * rng.standard_normal(D)).astype(np.float32)
  chains = [dict(X=torch.as_tensor(Xp, device=DEV), y=torch.as_tensor(y, device=DEV), D=D, n=n,
                 theta0=th0, key=(0, c), dkey=(3, c)) for c in range(2)]
  eng = fused.FusedGLM(chains, "logistic", mode, np.array([2e-3, 1e-3], np.float32), steps=2,
                       friction=0.5, target_bytes=n * 4 * Xp.shape[1] / nb)
  assert list(eng.nblocks_chain) == [nb, nb]
  if shift:  # records one float past an 8-byte boundary
    eng.partial = torch.zeros(eng.partial.numel() + 1, device=DEV)
    per = eng.partial.numel() // 2
    for c in range(2):
      eng._arr[c].partial = eng.partial.data_ptr() + 4 * (1 + c * per)
      assert eng._arr[c].partial % 8 == 4
    eng.table = torch.frombuffer(bytearray(bytes(eng._arr)), dtype=torch.uint8).to(DEV)
  return eng, om.Family("logistic", X, y), th0


@pytest.mark.parametrize("D,n,nb,shift", [
    (65, 70, 1, False), (65, 70, 2, False), (96, 1056, 17, False), (127, 1056, 33, False),
    (128, 512, 16, False), (129, 1056, 17, False), (256, 1056, 33, False), (257, 1056, 33, False),
    (33, 1056, 33, False), (5, 1056, 33, False), (1, 3, 1, False), (100, 1056, 17, True),
    (700, 1056, 33, False), (1023, 512, 16, False), (1024, 40, 2, True)])
@pytest.mark.parametrize("mode", ["sgld", "sghmc"])
def test_block_and_row_splits(D, n, nb, shift, mode):
  print(mode, D, n, nb, shift, flush=True)
  eng, fam, th0 = _engine(D, n, mode, nb, shift)
  eng.run(ITERS, loop=False)
  pot = lambda th, idx: om.stochastic_potential(fam, th, idx, 1.0)
  for c in range(2):
    key, dkey = np.array([0, c], np.uint32), np.array([3, c], np.uint32)
    eps = np.array([2e-3, 1e-3], np.float32)
    if mode == "sghmc":
      r = ost.sghmc(pot, th0, ITERS, eps, 2, 0.5, N, n, [D], key=key, dkey=dkey)
      _close(eng.momentum(c).cpu(), r["p"][-1], "momentum")
    else:
      r = ost.sgld(pot, th0, ITERS, eps, 1.0, N, n, [D], key=key, dkey=dkey)
      _close(eng.var[c].cpu(), r["variance"][-1], "var(lik)")
    _close(eng.theta(c).cpu(), r["theta"][-1], "theta")
    _close(eng.U[c].cpu(), r["U"][-1], "U")
    np.testing.assert_array_equal(R.key_words(eng.keys[c]), r["key"])
    np.testing.assert_array_equal(R.key_words(eng.dkeys[c]), r["dkey"])


@pytest.mark.parametrize("D", [65, 128, 129])
def test_loop_launch_of_the_wide_row_classes(D):
  """One-block chains in a loop launch give the bits of one launch per evaluation."""
  a, _, _ = _engine(D, 40, "sghmc", 1, False)
  b, _, _ = _engine(D, 40, "sghmc", 1, False)
  a.run(ITERS, loop=True)
  b.run(ITERS, loop=False)
  assert torch.equal(a.theta_flat, b.theta_flat) and torch.equal(a.mom_flat, b.mom_flat)
  assert torch.equal(a.U, b.U) and torch.equal(a.keys, b.keys)
