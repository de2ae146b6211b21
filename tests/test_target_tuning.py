"""The choice of the block-size tuners (CPU, simulated times): the default split is timed first
and stays unless a bytes-per-block target is faster by 1%."""
import pytest
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import fused  # noqa: E402


class Clock:
  """A table whose launches take the time of its split."""

  def __init__(self, cost, by_rule=True):
    self.cost, self.now, self.built = cost, 0.0, "default" if by_rule else 64 << 10
    e = object.__new__(fused.FusedGLM)
    e._default_target, e.prefer_loop, e.tuned = 64 << 10, None, None
    e.target_bytes = None if by_rule else 64 << 10
    e.loop_capable = lambda: False
    e._build_table, e._launch_steps = self.build, self.launch
    e._launch_iterations = lambda k: [self.launch() for _ in range(k)]
    e._snapshot, e._restore = dict, lambda s: None
    self.engine = e

  def build(self):
    e = self.engine
    self.built = "default" if e._blocks_by_rule else e.target_bytes
    # 1 MiB in blocks; a default split that no target gives
    e.nblocks_chain = [13 if e._blocks_by_rule else (1 << 20) // e.target_bytes]

  def launch(self):
    self.now += self.cost(self.built)


@pytest.mark.parametrize("default,best,kept", [(9.0, 10.0, True), (10.0, 9.95, True),
                                               (10.0, 9.0, False)])
def test_table_keeps_its_default_split(monkeypatch, default, best, kept):
  c = Clock(lambda split: default if split == "default" else best if split == 128 << 10 else 30.0)
  monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
  monkeypatch.setattr(fused.time, "perf_counter", lambda: c.now)
  tuned = c.engine.autotune(reps=2)
  assert c.built == ("default" if kept else 128 << 10)
  assert tuned["target_bytes"] == (None if kept else 128 << 10)
  assert tuned["seconds_per_iteration"] == pytest.approx(default if kept else best)
  assert c.engine.target_bytes == (64 << 10 if kept else 128 << 10)
  c.engine.autotune(candidates=[16 << 10, 32 << 10], reps=1)  # a caller's own candidates only
  assert c.built in (16 << 10, 32 << 10)


class Table:
  nblocks_chain = ()


def best_of(cost, candidates, tables, splits=None):
  """_best_targets over simulated costs; the split of a target is itself unless given."""
  engines = [Table() for _ in range(tables)]
  now = []

  def build(targets):
    now[:] = targets
    for e, tb in zip(engines, targets):
      e.nblocks_chain = [(splits or {}).get(tb, 0 if tb is None else tb)]
  return fused._best_targets(engines, candidates, build, lambda: cost[tuple(now)])


def test_tables_of_a_group_choose_one_by_one():
  cost = {(None, None): 10.0, (1, 1): 9.95, (2, 2): 12.0, (None, 1): 9.8, (None, 2): 11.0,
          (1, None): 12.0, (2, None): 13.0, (2, 1): 13.0}
  assert best_of(cost, [None, 1, 2], 2) == (9.8, [None, 1])
  assert best_of({(2,): 1.001, (1,): 1.0}, [2, 1], 1) == (1.0, [1])


def test_a_target_with_the_default_split_is_not_timed_again():
  cost = {(None,): 10.0, (1,): 9.0, (2,): 11.0}
  assert best_of(cost, [None, 1, 2], 1, {None: 4, 1: 4, 2: 8}) == (10.0, [None])


def test_a_slow_first_timing_does_not_cost_the_default_split():
  """The clocks settle while the default split is timed: it is timed again against the best
  target."""
  e, now, count = Table(), [], [0]

  def build(targets):
    now[:] = targets
    e.nblocks_chain = [0 if targets[0] is None else targets[0]]

  def timed():
    count[0] += 1
    return (10.0 if now[0] is None else 10.1) * (1.2 if count[0] <= 4 else 1.0)
  assert fused._best_targets([e], [None, 1, 2], build, timed) == (10.0, [None])


def test_candidates():
  by_rule, by_bytes = Clock(None).engine, Clock(None, False).engine
  assert fused._target_candidates([by_rule])[0] is None
  assert None not in fused._target_candidates([by_bytes])
  assert fused._target_candidates([by_bytes, by_rule])[0] is None
  assert 64 << 10 in fused._target_candidates([by_rule])
