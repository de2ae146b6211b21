"""sgmc_glm_blocks(n, D), the block count that callers of the minibatch potentials are sent
to, fits the static scratch of sgmc_glm_potential_noalloc (262,080 record floats) wherever
blocks of 4096 rows do (CPU), and the no-allocation potential runs with it (GPU)."""
import pytest
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import _lib as L  # noqa: E402

SCRATCH = 262_080
ROWS = 4096  # likelihoods a block stages


@pytest.mark.parametrize("D", [1, 64, 256, 257, 500, 508, 509, 511, 512, 513, 1020, 1021, 1024])
def test_recommended_blocks_fit_the_scratch(D):
  record = 4 * ((D + 3) // 4) + 2
  for n in list(range(1, 70_000, 251)) + [8160, 8161, 16_288, 16_289, 100_000, 1_000_000,
                                          2_147_483_647]:
    nb = int(L.query("sgmc_glm_blocks", n, D))
    assert 1 <= nb <= n and nb * ROWS >= n
    assert nb * record <= SCRATCH or nb == -(-n // ROWS)


@pytest.mark.gpu
@pytest.mark.parametrize("n,D", [(16_289, 512), (40_001, 509), (8161, 1024), (60_000, 1021)])
def test_noalloc_runs_with_the_recommended_blocks(n, D):
  print("noalloc", n, D, flush=True)
  nb = int(L.query("sgmc_glm_blocks", n, D))
  g = torch.Generator(device="cuda").manual_seed(n + D)
  ld = (D + 3) // 4 * 4
  X = torch.randn((n, ld), generator=g, device="cuda") / D ** 0.5
  y = (torch.rand(n, generator=g, device="cuda") < 0.5).float()
  w = 0.3 * torch.randn(D, generator=g, device="cuda")
  outs = []
  for noalloc in (False, True):
    U, grad = torch.empty(1, device="cuda"), torch.empty(D, device="cuda")
    args = [L.LIK_LOGISTIC, L.ptr(X), ld, L.ptr(y), None, n, 2 * n, D, L.ptr(w), 1.0, 1, 1.0, 1.0,
            L.ptr(U), L.ptr(grad), None, None]
    if noalloc:
      L.call("sgmc_glm_potential_noalloc", *args, nb, L.stream())
    else:
      ws = torch.zeros(int(L.query("sgmc_glm_workspace_floats", n, D, nb)), device="cuda")
      L.call("sgmc_glm_potential", *args, L.ptr(ws), ws.numel(), nb, L.stream())
    outs.append(torch.cat([U, grad]))
  assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
