"""The default split of tables of many equal chains (host rule, CPU): the blocks fill the
compute units' rounds, and no block is so long that its rows' latency outlasts the table's
stream."""
import math

import pytest

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import fused  # noqa: E402

CUS = 256


@pytest.mark.parametrize("D", [300, 512, 1000])
@pytest.mark.parametrize("n", [2048, 4096])
def test_last_round_is_filled(D, n):
  """A few blocks past a full round would leave most units idle for a second one."""
  for C in [*range(17, 100, 3), *range(100, 700, 17)]:
    nb = fused.default_blocks([n] * C, [D] * C, True, CUS)[0]
    rounds = C * nb / CUS
    assert rounds / math.ceil(rounds) >= 0.79, (C, nb)


@pytest.mark.parametrize("D,C,n,least,most", [
    (300, 171, 4096, 4, 8), (300, 300, 4096, 3, 8), (200, 500, 4096, 2, 8), (512, 171, 2048, 3, 8),
    (1000, 55, 4096, 4, 4), (512, 55, 4096, 4, 4), (1000, 500, 4096, 1, 1), (512, 230, 4096, 1, 1)])
def test_measured_splits(D, C, n, least, most):
  """Counts of which the neighbours measured slower than the split before (blocks of 64 KiB or
  1/2048 of the table)."""
  assert least <= fused.default_blocks([n] * C, [D] * C, True, CUS)[0] <= most


@pytest.mark.parametrize("n,D,loops,want", [
    ([128], [100], True, [1]),                # 51 KiB alone: a loop launch
    ([128], [100], False, [4]),               # the same without one
    ([128, 4096], [100, 512], True, [3, 128]),  # beside a chain of several blocks
    ([128, 128, 64], [100, 100, 30], True, [1, 1, 1])])
def test_the_line_of_loop_launches_needs_them(n, D, loops, want):
  assert fused.table_blocks(n, D, loops, CUS) == want
