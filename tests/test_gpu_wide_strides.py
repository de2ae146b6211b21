"""Row strides and layer widths at which byte offsets leave 31 bits (GPU, up to about 100 GB
of device memory)."""
import numpy as np
import pytest
import torch

from oracle import model as om

from jax_sgmc_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _last_split_stride(D):
  """The longest stride whose tile of 32 rows the split kernel reaches."""
  return (2 ** 31 - 1 - 16 * ((D + 3) // 4)) // 124 // 4 * 4


@pytest.mark.parametrize("D,C,over", [(5, 3, 0), (5, 3, 4), (40, 33, 0), (300, 4, 100_000),
                                      (17, 3, 2_000_000)])
def test_split_full_potential_of_a_wide_matrix(D, C, over):
  """The rows are a column slice of a wide matrix: 33 rows (a tile and one row) at the
  longest stride of the split kernel and at longer ones. As for every split full potential
  2e-6 relative to float64."""
  ldx, N = _last_split_stride(D) + over, 33
  print("split full potential, stride", ldx, "D", D, "chains", C, flush=True)
  rng = np.random.default_rng(D + C)
  X = (rng.standard_normal((N, D)) / np.sqrt(D)).astype(np.float32)
  y = (rng.random(N) < 0.5).astype(np.float32)
  th = (0.5 * rng.standard_normal((C, D))).astype(np.float32)
  wide = torch.zeros((N, ldx), device=DEV)
  wide[:, :D] = torch.as_tensor(X, device=DEV)
  yd, thd = torch.as_tensor(y, device=DEV), torch.as_tensor(th, device=DEV)
  nb = 3
  ws = torch.zeros(int(L.query("sgmc_glm_full_chains_workspace_doubles", nb)), device=DEV,
                   dtype=torch.float64)
  out = torch.empty(C, dtype=torch.float64, device=DEV)
  z = X.astype(np.float64) @ th.astype(np.float64).T
  lik = y[:, None] * z - np.logaddexp(0, z)
  for _ in range(2):
    L.call("sgmc_glm_full_potential_chains_split", L.LIK_LOGISTIC, L.ptr(wide), ldx, L.ptr(yd), N,
           D, L.ptr(thd), D, C, 0.7, 1, 2.0, 1.5, 14 - int(np.frexp(np.abs(X).max())[1]),
           L.ptr(out), L.ptr(ws), ws.numel(), nb, L.stream())
    got = out.cpu().numpy()
    for c in range(C):
      want = (-np.sum(lik[:, c]) - om.gaussian_logprior(th[c], 2.0)[0]) / 1.5
      assert abs(got[c] - want) <= 2e-6 * abs(want), (c, got[c], want)
