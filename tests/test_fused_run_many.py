"""sgmc_glm_fused_run with more tables than one call takes in turn: each is checked before any
launch (CPU), and each gives what it gives alone (GPU)."""
import ctypes

import numpy as np
import pytest
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import _lib as L  # noqa: E402
from jax_sgmc_amd import fused  # noqa: E402


def test_every_table_is_checked():
  runs = (L.GlmRun * 200)()
  codes = (ctypes.c_int32 * 2)(L.OP_ITERATIONS, 0)
  for r in runs:
    for f in ("chains", "eps_table", "iter", "done"):
      setattr(r, f, 16)
    r.nchains, r.nblocks, r.table_len, r.steps, r.pot_temperature = 1, 1, 1, 1, 1.0
    r.ops, r.nops = ctypes.addressof(codes), 1
  L.call("sgmc_glm_fused_run", runs, 200)
  runs[199].mode = 6
  with pytest.raises(ValueError, match="mode"):
    L.call("sgmc_glm_fused_run", runs, 200)


@pytest.mark.gpu
def test_many_tables_equal_single_tables():
  print("70 tables in one call", flush=True)
  g = torch.Generator(device="cuda").manual_seed(5)
  X = torch.randn((500, 12), generator=g, device="cuda")
  y = torch.randn(500, generator=g, device="cuda")

  def table(k):
    return fused.FusedGLM([dict(X=X, y=y, D=11, n=100 + k, theta0=np.zeros(11, np.float32),
                                key=(1, k), dkey=(2, k))], "linear_gaussian", "sgld",
                          np.full(8, 1e-4, np.float32), target_bytes=2000)
  many, alone = [table(k) for k in range(70)], [table(k) for k in range(70)]
  fused._execute_tables([(e, None, [("it",)] * 3) for e in many])
  for e in alone:
    for _ in range(3):
      e._launch_steps()
  torch.cuda.synchronize()
  for a, b in zip(many, alone):
    assert a.iteration_count() == 3
    assert torch.equal(a.theta_flat, b.theta_flat) and torch.equal(a.keys, b.keys)
