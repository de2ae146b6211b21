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


def test_tables_of_a_group_choose_one_by_one():
  cost = {(None, None): 10.0, (1, 1): 9.95, (2, 2): 12.0, (None, 1): 9.8, (None, 2): 11.0,
          (1, None): 12.0, (2, None): 13.0, (2, 1): 13.0}
  assert fused._best_targets(2, [None, 1, 2], lambda t: cost[tuple(t)]) == (9.8, [None, 1])
  assert fused._best_targets(1, [2, 1], lambda t: {1: 1.0, 2: 1.001}[t[0]]) == (1.0, [1])


def test_candidates():
  by_rule, by_bytes = Clock(None).engine, Clock(None, False).engine
  assert fused._target_candidates([by_rule])[0] is None
  assert None not in fused._target_candidates([by_bytes])
  assert fused._target_candidates([by_bytes, by_rule])[0] is None
  assert 64 << 10 in fused._target_candidates([by_rule])
