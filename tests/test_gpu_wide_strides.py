"""Row strides and layer widths at which byte offsets leave 31 bits (GPU, up to about 100 GB
of device memory)."""
import numpy as np
import pytest
import torch

from oracle import model as om
from oracle import steps as ost

from jax_sgmc_amd import _lib as L
from jax_sgmc_amd import mlp as M

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


@pytest.mark.parametrize("dims", [(17_400_000, 128, 128), (64, 17_400_064, 128)])
def test_wide_mlp_layers(dims):
  """The float32 gradient and a plain SGLD update without noise of a net with a layer of
  17.4 M: 31 rows of it span more than 2^31 bytes, as rows of an activation (G1's and G2's
  left operand) and as rows of a weight's state (gW1 and gW2). The whole gradient at
  1e-4 in norm of the float64 one, as for every float32 gradient; the update within an ulp of theta plus the
  roundings of its step."""
  D, H1, H2 = dims
  n = N = 64
  print("MLP layers", dims, flush=True)
  g = torch.Generator(device=DEV).manual_seed(3)
  X = torch.rand((N, D), generator=g, device=DEV) - 0.5
  labels = torch.randint(0, 10, (N,), generator=g, device=DEV, dtype=torch.int32)
  P = M.param_count(D, H1, H2)
  eps = 1e-3
  eng = M.FusedMLP(X, labels, dims, n, np.zeros((1, P), np.float32), np.full(2, eps, np.float32),
                   dkeys=np.array([[2, 5]], np.uint32), precision="fp32", noise_temperature=0.0)
  off = 0
  for rows, cols in ((D, H1), (H1, H2), (H2, 10)):
    eng.theta[0, off:off + rows * cols].normal_(0.0, (2.0 / rows) ** 0.5, generator=g)
    off += rows * cols
  _, grad = eng.potential_and_grad()
  eng.grad = None
  th0 = eng.theta.clone()
  print("update", flush=True)
  eng.iteration()
  for k in range(0, P, 1 << 28):
    part = slice(k, k + (1 << 28))
    t, step = th0[0, part], eps * grad[0, part]
    off = (eng.theta[0, part] - (t - step)).abs_()
    assert bool((off <= 2.0 ** -23 * (t.abs() + 3.0 * step.abs())).all()), k
  print("reference", flush=True)
  _, idx = ost.draw_indices(np.array([2, 5], np.uint32), N, n)
  idx = torch.as_tensor(np.asarray(idx).astype(np.int64), device=DEV)
  x, lab = X[idx].double(), labels[idx].long()
  th = [p.double() for p in _leaves(th0[0], dims)]
  h1 = torch.relu(x @ th[0] + th[3])
  h2 = torch.relu(h1 @ th[1] + th[4])
  logp = torch.log_softmax(h2 @ th[2] + th[5], dim=1)
  dL = (-N / n) * (torch.nn.functional.one_hot(lab, 10).double() - logp.exp())
  dA2 = (dL @ th[2].T) * (h2 > 0)
  dA1 = (dA2 @ th[1].T) * (h1 > 0)
  ref = [lambda: x.T @ dA1, lambda: h1.T @ dA2, lambda: h2.T @ dL, lambda: dA1.sum(0),
         lambda: dA2.sum(0), lambda: dL.sum(0)]
  size = diff = 0.0
  for r, t, got in zip(ref, th, _leaves(grad[0], dims)):
    r = r().add_(t)
    size += r.norm().item() ** 2
    diff += r.sub_(got).norm().item() ** 2
  print("error in norm", (diff / size) ** 0.5, flush=True)
  assert diff <= 1e-8 * size


def _leaves(flat, dims):
  D, H1, H2 = dims
  out, off = [], 0
  for shape in ((D, H1), (H1, H2), (H2, 10), (H1,), (H2,), (10,)):
    size = int(np.prod(shape))
    out.append(flat[off:off + size].reshape(shape))
    off += size
  return out
