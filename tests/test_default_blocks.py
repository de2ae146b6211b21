"""The default split of a chain table into grid blocks (host rule, CPU)."""
import numpy as np
import pytest

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import fused  # noqa: E402


@pytest.mark.parametrize("C,D,n,loops,blocks", [
    (64, 512, 4096, True, 4), (32, 512, 4096, True, 8), (16, 100, 1000, True, 16),
    (64, 256, 512, True, 8), (64, 100, 2048, False, 8), (1, 32, 128, True, 1),
    (1, 32, 128, False, 1), (1, 100, 128, True, 1), (1, 100, 128, False, 4),
    (1, 512, 4096, True, 128), (1, 12, 4096, True, 16), (1000, 512, 4096, True, 1),
    (1000, 3, 20000, True, 5)])
def test_uniform_tables(C, D, n, loops, blocks):
  assert fused.default_blocks([n] * C, [D] * C, loops, 256) == [blocks] * C


def test_every_split_is_legal():
  """Each block has a row and at most LDS_ROWS of them, over random mixed tables."""
  rng = np.random.default_rng(0)
  for _ in range(300):
    C = int(rng.integers(1, 70))
    n = np.exp(rng.uniform(0, np.log(60000), C)).astype(int) + 1
    D = np.exp(rng.uniform(0, np.log(1024), C)).astype(int).clip(1, 1024)
    for loops in (True, False):
      nb = fused.default_blocks(n, D, loops, 256)
      assert all(1 <= b <= k and -(-k // b) <= fused.LDS_ROWS for b, k in zip(nb, n))
