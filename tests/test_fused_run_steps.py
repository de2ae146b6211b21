"""SGMC_OP_ITERATIONS of sgmc_glm_fused_run with `steps` set on a table whose mode has no
leapfrog steps (GPU): an iteration is one evaluation, as in a loop launch."""
import ctypes

import numpy as np
import pytest
import torch

from jax_sgmc_amd import _lib as L
from jax_sgmc_amd import fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["sgld", "sgld_rms"])
@pytest.mark.parametrize("op,target", [(L.OP_ITERATIONS, 4000), (L.OP_LOOP, 1 << 30)])
def test_iterations_of_modes_without_steps(mode, op, target):
  print(mode, op, flush=True)
  g = torch.Generator(device="cuda").manual_seed(4)
  X = torch.randn((500, 12), generator=g, device="cuda")
  y = torch.randn(500, generator=g, device="cuda")

  def table():
    return fused.FusedGLM([dict(X=X, y=y, D=11, n=400, theta0=np.zeros(11, np.float32), key=(1, c),
                                dkey=(2, c)) for c in range(3)], "linear_gaussian", mode,
                          np.full(16, 1e-4, np.float32), target_bytes=target)
  one, many = table(), table()
  for e, steps in ((one, 1), (many, 3)):
    codes = (ctypes.c_int32 * 2)(op, 4)
    r = e._run_desc(codes, torch.cuda.current_stream().cuda_stream)
    r.steps = steps
    L.call("sgmc_glm_fused_run", (L.GlmRun * 1)(r), 1)
  torch.cuda.synchronize()
  assert one.iteration_count() == many.iteration_count() == 4
  assert torch.equal(one.theta_flat, many.theta_flat) and torch.equal(one.keys, many.keys)
