"""Rounding of the float32 sums over the rows of one long block (GPU): 4096 equal terms
t = 1 + 2^-15 - 2^-23, which a running sum rounds down at every addition once it is past 512
(2e-5 relative after a wavefront's 1024; a lane that shares them with others, at D <= 128, adds
at most 512). Sums of 64 rows, added up, stay within (64 + 16 + 4 + 8) 2^-24 = 5.5e-6: at most
64 additions of a lane in a chunk, 16 chunks of a wavefront, 4 wavefronts, the scaling."""
import pytest
import torch

from jax_sgmc_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [8, 24, 50, 100, 200, 300, 600])
def test_gradient_of_one_long_block(D):
  print("one block of 4096 rows, D", D, flush=True)
  n, ld = 4096, (D + 3) // 4 * 4
  t = 1.0 + 2.0 ** -15 - 2.0 ** -23
  X = torch.zeros((n, ld), device=DEV)
  X[:, :D] = 1.0
  y = torch.full((n,), t, device=DEV)
  assert y[0].item() == t
  w = torch.zeros(D, device=DEV)
  U, g = torch.empty(1, device=DEV), torch.empty(D, device=DEV)
  ws = torch.zeros(int(L.query("sgmc_glm_workspace_floats", n, D, 1)), device=DEV)
  # theta = 0, sigma = 1: each row adds (y - 0) / 1 to every column
  L.call("sgmc_glm_potential", L.LIK_LINEAR_GAUSSIAN, L.ptr(X), ld, L.ptr(y), None, n, n, D,
         L.ptr(w), 1.0, 0, 1.0, 1.0, L.ptr(U), L.ptr(g), None, None, L.ptr(ws), ws.numel(), 1,
         L.stream())
  want = -n * t
  assert ((g.double() - want).abs() <= (64 + 16 + 4 + 8) * 2.0 ** -24 * abs(want)).all(), \
      (g[0].item(), want)
