"""A TableGroup whose tables live on another device than the caller's current one (CPU, with
stand-ins for torch's streams and devices): the launches are issued under the tables' device,
and the tables' streams are forked from and joined to the caller's stream by events, since
the null stream of one device orders nothing on another."""
import contextlib

import numpy as np
import pytest
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import fused  # noqa: E402


class Stream:
  def __init__(self, device, handle, log):
    self.device, self.cuda_stream, self.log = torch.device("cuda", device), handle, log

  def wait_stream(self, other):
    self.log.append(("wait", self.device.index, self.cuda_stream, other.device.index,
                     other.cuda_stream))


class Engine:
  host_iter = 0

  def _loop_arg(self, loop):
    return False

  def _plan(self, iterations, loop):
    return [("it",)] * iterations


@pytest.mark.parametrize("current,handle,events", [(0, 0, True), (1, 0, False), (1, 7, True),
                                                   (0, 7, True)])
@pytest.mark.parametrize("call", ["run", "iteration"])
def test_launches_under_the_tables_device(monkeypatch, current, handle, events, call):
  log = []
  device = [current]

  @contextlib.contextmanager
  def under(d):
    d = torch.device(d)
    before, device[0] = device[0], d.index
    yield
    device[0] = before
  caller = {d: Stream(d, handle if d == current else 0, log) for d in (0, 1)}
  monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: caller[device[0]])
  monkeypatch.setattr(torch.cuda, "device", under)
  monkeypatch.setattr(fused, "_execute_tables",
                      lambda items: log.append(("launch", device[0], [i[1] for i in items])))
  grp = object.__new__(fused.TableGroup)
  grp.engines, grp.stream_of = [Engine(), Engine()], [0, 1]
  grp.streams = [Stream(1, 11, log), Stream(1, 12, log)]
  grp.offsets = np.array([0, 1, 2])
  grp.run(3) if call == "run" else grp.iteration()
  launch = ("launch", 1, grp.streams)
  fork = [("wait", 1, h, current, handle) for h in (11, 12)]
  join = [("wait", current, handle, 1, h) for h in (11, 12)]
  assert log == (fork + [launch] + join if events else [launch])
  assert device[0] == current
