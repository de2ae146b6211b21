"""sgmc_glm_fused_run (CPU-only checks): the ctypes mirror of its argument struct has the C
layout, bad tables are refused before any launch, and plans are grouped into native runs.
That its launches give the per-launch results is covered by every engine test on the GPU,
and test_interleaved_tables_equal_single_tables here."""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

import __graft_entry__

__graft_entry__.load()

from jax_sgmc_amd import _lib as L  # noqa: E402
from jax_sgmc_amd import fused  # noqa: E402

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_run_struct_layout(tmp_path):
  lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "sgmc.h"', "int main(void) {",
           'printf("%zu\\n", sizeof(sgmc_glm_run));']
  lines += [f'printf("%zu\\n", offsetof(sgmc_glm_run, {f}));' for f, _ in L.GlmRun._fields_]
  src, exe = tmp_path / "l.c", tmp_path / "l"
  src.write_text("\n".join(lines + ["return 0; }"]))
  subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)],
                 check=True)
  got = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True,
                                        text=True).stdout.split()]
  assert got == [ctypes.sizeof(L.GlmRun)] + [getattr(L.GlmRun, f).offset
                                             for f, _ in L.GlmRun._fields_]


def run_of(**kw):
  """A table that passes the checks (no launch: no operations)."""
  r = L.GlmRun(chains=16, eps_table=16, iter=16, done=16, nchains=2, nblocks=4,
               uniform_dclass=0, family=0, has_prior=1, mode=L.MODE_SGLD, steps=1, table_len=1,
               sigma=1.0, prior_scale=1.0, pot_temperature=1.0)
  ops = kw.pop("ops", [])
  r._codes = (ctypes.c_int32 * max(1, len(ops)))(*ops)
  r.ops, r.nops = ctypes.addressof(r._codes), len(ops) // 2
  for k, v in kw.items():
    setattr(r, k, v)
  return r


@pytest.mark.parametrize("bad", [dict(chains=None), dict(eps_table=None), dict(iter=None),
                                 dict(done=None), dict(nblocks=3), dict(nchains=0),
                                 dict(nblocks=1), dict(table_len=0), dict(nops=-1),
                                 dict(ops=[0, -1]), dict(ops=[3, 1]), dict(ops=[-1, 1]),
                                 dict(ops=[L.OP_LOOP, 1]),
                                 dict(ops=[L.OP_LOOP, 1], nblocks=2, mode=L.MODE_SGGMC),
                                 dict(ops=[L.OP_SWAP, 1]),
                                 dict(ops=[L.OP_SWAP, 1], pairs=16, npairs=1),
                                 dict(ops=[L.OP_SWAP, 1], pairs=16, swap_every=1),
                                 dict(family=2), dict(mode=6), dict(mode=-1), dict(steps=0),
                                 dict(pot_temperature=0.0)])
def test_bad_tables_are_refused(bad):
  # the second table's fault is found before the first table's launches
  good, poor = run_of(ops=[L.OP_ITERATIONS, 0, L.OP_LOOP, 0], nblocks=2), run_of(**bad)
  arr = (L.GlmRun * 2)(good, poor)
  with pytest.raises(ValueError):
    L.call("sgmc_glm_fused_run", arr, 2)
  with pytest.raises(ValueError):
    L.call("sgmc_glm_fused_run", arr, 0)
  L.call("sgmc_glm_fused_run", (L.GlmRun * 1)(good), 1)


def test_plans_are_cut_into_native_runs():
  it, seg = ("it",), lambda ops: [tuple(s) for s in fused._segments(ops)]
  I, Lp, S = L.OP_ITERATIONS, L.OP_LOOP, L.OP_SWAP
  assert seg([]) == []
  assert seg([it, it, ("swap",), it]) == [("native", [I, 2, S, 1, I, 1], 3)]
  assert seg([("loop", 7), ("swap",), ("loop", 3)]) == [("native", [Lp, 7, S, 1, Lp, 3], 10)]
  assert seg([it, ("mh",), it, it, ("mh",)]) == [("native", [I, 1], 1), ("mh",),
                                                 ("native", [I, 2], 2), ("mh",)]
  k = fused._RUN_ITERATIONS
  assert seg([it] * (2 * k + 1)) == [("native", [I, k], k), ("native", [I, k], k),
                                     ("native", [I, 1], 1)]
  assert seg([("loop", k), ("loop", k)]) == [("native", [Lp, k], k), ("native", [Lp, k], k)]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["sgld_rms", "sghmc", "obabo"])
def test_interleaved_tables_equal_single_tables(mode):
  """Tables of different sizes and iteration lengths run side by side through one native
  call give what each gives launched one evaluation at a time."""
  g = torch.Generator(device="cuda").manual_seed(1)
  X = torch.randn((3000, 24), generator=g, device="cuda")
  y = (torch.rand(3000, generator=g, device="cuda") < 0.5).float()

  def table(C, n):
    chains = [dict(X=X, y=y, D=23, n=n, theta0=np.zeros(23, np.float32), key=(1, c),
                   dkey=(2, c)) for c in range(C)]
    return fused.FusedGLM(chains, "logistic", mode, np.full(8, 1e-4, np.float32), steps=2,
                          friction=0.5, target_bytes=6000)
  group = fused.TableGroup([table(3, 200), table(5, 331)])
  alone = [table(3, 200), table(5, 331)]
  group.run(5)
  for e in alone:
    for _ in range(5):
      e._launch_steps()
  torch.cuda.synchronize()
  for a, b in zip(group.engines, alone):
    assert a.host_iter == 5 and a.iteration_count() == 5
    assert torch.equal(a.theta_flat, b.theta_flat) and torch.equal(a.U, b.U)
    assert torch.equal(a.keys, b.keys) and torch.equal(a.dkeys, b.dkeys)


@pytest.mark.gpu
def test_group_runs_are_ordered_with_the_callers_stream():
  """A group's tables run on streams of their own. Work of the caller's stream before
  and after a run is ordered with it without events on the null stream: eager work there,
  another (non-blocking) stream that waits for it, host reads; and with events where the
  caller is on another stream."""
  g = torch.Generator(device="cuda").manual_seed(2)
  X = torch.randn((40000, 256), generator=g, device="cuda")
  y = (torch.rand(40000, generator=g, device="cuda") < 0.5).float()

  def group():
    mk = lambda k: fused.FusedGLM(
        [dict(X=X, y=y, D=256, n=4096, theta0=np.zeros(256, np.float32), key=(k, c),
              dkey=(7, c)) for c in range(8)], "logistic", "sgld",
        np.full(8, 1e-6, np.float32))
    return fused.TableGroup([mk(1), mk(2)])
  want = group()
  for e in want.engines:
    for _ in range(60):
      e._launch_steps()
  torch.cuda.synchronize()
  want = [e.theta_flat.clone() for e in want.engines]
  for where in ("null", "side", "other"):
    grp, side, other = group(), torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    got = [torch.empty_like(w) for w in want]
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side if where == "side" else torch.cuda.current_stream()):
      for e in grp.engines:  # earlier work of the caller: a start the run must see
        e.theta_flat.fill_(5.0)
        e.theta_flat.zero_()
      grp.run(60)
      if where == "other":
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
          for a, e in zip(got, grp.engines):
            a.copy_(e.theta_flat)
        other.synchronize()
      else:
        for a, e in zip(got, grp.engines):
          a.copy_(e.theta_flat)
        torch.cuda.current_stream().synchronize()
      host = [a.cpu() for a in got]
    for w, h in zip(want, host):
      assert torch.equal(w.cpu(), h), where
