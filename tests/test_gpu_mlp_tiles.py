"""Tile edges of the MLP engine's GEMMs and head (GPU).

Potential and gradient at shapes that reach every tile and split of the GEMMs and their
remainders: K below one stage, K / splits that ends inside a stage (a half stage of e4m3 is
64 values, of bf16 32), an odd number of stages, one to four groups over K, and the largest
tile (256 x 128, 16 chains). The reference is the evaluation in float64 with the operands
rounded where the engine rounds them (bf16, or e4m3 at the engine's scales; nowhere for
float32): what is left is float32 accumulation and, layer by layer, the operands that its
differences move over a rounding boundary. Tolerances: the engine's at its benchmark shapes
(potential / gradient in norm: float32 1e-5 / 1e-4, bf16 1e-2 / 3e-2, e4m3 3e-2 / 0.15); a
wrong element is an error of order one."""
import numpy as np
import pytest
import torch

from oracle import model as om
from oracle import steps as ost

from jax_sgmc_amd import mlp as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
N = 2048
TOL = {"fp32": (1e-5, 1e-4), "bf16": (1e-2, 3e-2), "fp8": (3e-2, 0.15)}

# (D_in, H1, H2), n, chains, groups over K of G1, G2, G3 (0: the built-in choice)
SHAPES = [
    ((64, 128, 128), 64, 1, (1, 1, 1)),        # K of one half stage (e4m3)
    ((192, 128, 256), 64, 3, (2, 2, 2)),       # K / 2 ends inside a stage
    ((448, 256, 128), 192, 2, (1, 2, 1)),      # odd number of stages, n not a tile of 128
    ((192, 384, 384), 64, 1, (3, 3, 3)),       # three groups
    ((256, 256, 512), 128, 2, (4, 4, 4)),      # four groups
    ((128, 512, 512), 256, 8, (0, 0, 0)),      # 64 x 128 tiles
    ((64, 1024, 1024), 512, 16, (1, 1, 1)),    # 256 x 128 tiles; the head's largest blocks
    ((64, 1024, 1024), 384, 22, (1, 1, 1)),    # 128 x 128 tiles
    ((128, 128, 384), 256, 16, (0, 0, 0)),     # the head at 4096 rows, columns in twos at the end
    ((64, 128, 1536), 64, 2, (0, 0, 0)),       # the head with W3 past its LDS
]


def tune_of(precision, dims, splits):
  """tune[] codes of the activation GEMMs with the given groups over K (the smallest k-tile
  of the precision, so that K fits)."""
  bk = {"fp32": 32, "bf16": 32, "fp8": 64}[precision]
  K = (dims[0], dims[1], dims[2])
  return [bk * 16 + s if s and k % (bk * s) == 0 else 0 for k, s in zip(K, splits)] + [0, 0]


def rounded_reference(precision, X, labels, dims, theta, q):
  """(U, gradient) of one chain on the rows X in float64, prior scale 1, operands rounded."""
  f64 = torch.float64
  bf16 = lambda v: torch.as_tensor(v).float().bfloat16().to(f64)

  def e4m3(v, scale):
    v32 = (torch.as_tensor(v).float() * float(scale)).clamp(-448.0, 448.0)
    return v32.to(torch.float8_e4m3fn).to(f64) / float(scale)

  if precision == "fp32":
    r = [lambda v: torch.as_tensor(v).to(f64)] * 6
  elif precision == "bf16":
    r = [bf16] * 6
  else:  # scale words: X, h1, dA2, dA1, W1, W2
    r = [lambda v, k=k: e4m3(v, q[k]) for k in range(6)]
  h2r = r[1] if precision == "fp32" else bf16
  W1, W2, W3, b1, b2, b3 = [torch.as_tensor(np.ascontiguousarray(t)).to(f64)
                            for t in om.mlp_unflatten(theta, dims + (10,))]
  x, w1, w2 = r[0](X), r[4](W1), r[5](W2)
  h1 = r[1](torch.relu(x @ w1 + b1))
  h2 = h2r(torch.relu(h1 @ w2 + b2))
  logp = torch.log_softmax(h2 @ W3 + b3, dim=1)
  lab = torch.as_tensor(labels).long()
  n = X.shape[0]
  lik = logp[torch.arange(n), lab].sum()
  onehot = torch.nn.functional.one_hot(lab, 10).to(f64)
  dL = (-N / n) * (onehot - logp.exp())
  dA2 = r[2]((dL @ W3.T) * (h2 > 0))
  dA1 = r[3]((dA2 @ w2.T) * (h1 > 0))
  parts = [x.T @ dA1, h1.T @ dA2, h2.T @ dL, dA1.sum(0), dA2.sum(0), dL.sum(0)]
  t = torch.as_tensor(theta).to(f64)
  prior = -0.5 * (t * t + np.log(2 * np.pi)).sum()
  g = torch.cat([p.reshape(-1) for p in parts]) + t
  return float(-(N / n) * lik - prior), g.numpy()


@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp8"])
@pytest.mark.parametrize("dims,n,C,splits", SHAPES)
def test_potential_and_gradient_at_tile_edges(dims, n, C, splits, precision):
  print("MLP tiles:", precision, dims, n, C, splits, flush=True)
  rng = np.random.default_rng(5)
  X = rng.random((N, dims[0]), dtype=np.float32)
  labels = rng.integers(0, 10, N).astype(np.int32)
  th = np.stack([M.init_params(60 + c, *dims) for c in range(C)])
  dkeys = np.array([[2, 5 + c] for c in range(C)], np.uint32)
  eng = M.FusedMLP(torch.as_tensor(X, device=DEV), torch.as_tensor(labels, device=DEV), dims, n,
                   th, np.full(4, 1e-5, np.float32),
                   keys=np.array([[0, 1 + c] for c in range(C)], np.uint32), dkeys=dkeys,
                   prior_scale=1.0, precision=precision, tune=tune_of(precision, dims, splits))
  scales = eng.q.cpu().numpy() if precision == "fp8" else [None] * C
  U, g = eng.potential_and_grad()
  torch.cuda.synchronize()
  for c in sorted({0, C - 1}):
    _, idx = ost.draw_indices(dkeys[c], N, n)
    Ur, gr = rounded_reference(precision, X[idx], labels[idx], dims, th[c], scales[c])
    gc = g[c].cpu().numpy().astype(np.float64)
    assert abs(U[c].item() - Ur) <= TOL[precision][0] * abs(Ur)
    assert np.linalg.norm(gc - gr) < TOL[precision][1] * np.linalg.norm(gr)
