"""The MLP engine's tuning candidates name one code per choice that reaches a kernel (CPU,
host plan only): the split-K factors of the forward GEMMs that fit their K, and one code for
each parameter GEMM."""
import pytest

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import mlp as M  # noqa: E402


@pytest.mark.parametrize("precision,dims,n,splits", [
    ("bf16", (3072, 512, 512), 256, [[1, 2, 3, 4], [1, 2, 4], [1, 2, 4], [1], [1]]),
    ("fp8", (3072, 1024, 1024), 512, [[1, 2, 3, 4], [1, 2, 4], [1, 2, 4], [1], [1]]),
    ("fp32", (384, 256, 128), 64, [[1, 2, 3, 4], [1, 2, 4], [1, 2, 4], [1], [1]]),
    ("bf16", (192, 128, 128), 64, [[1, 2, 3], [1, 2, 4], [1, 2, 4], [1], [1]]),
    ("fp8", (192, 128, 128), 64, [[1, 3], [1, 2], [1, 2], [1], [1]])])
def test_one_candidate_per_split(precision, dims, n, splits):
  eng = object.__new__(M.FusedMLP)
  eng.dims, eng.n, eng.C, eng.precision, eng.tune = dims, n, 4, precision, [0] * 5
  builtin = [k * 16 + s for k, s in eng.gemm_plan()]
  for slot in range(5):
    codes = eng.tile_candidates(slot)
    assert [c & 15 for c in codes] == splits[slot]
    assert builtin[slot] in codes
    for code in codes:  # each is accepted
      eng.tune = [0] * 5
      eng.tune[slot] = code
      eng.gemm_plan()
    eng.tune = [0] * 5
