"""Lanes of one wavefront hand data to each other through LDS behind wave_sync, whose fences
hold the compiler (CPU, on the sources): a bare wave barrier orders the schedule and is no
memory fence, so what lies beyond it may be moved across by an optimiser that sees no
dependence between lanes."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-sgmc_amd",
                    "csrc")


def test_wave_barriers_are_fenced():
  bare = {}
  for name in sorted(os.listdir(CSRC)):
    with open(os.path.join(CSRC, name)) as f:
      code = re.sub(r"//[^\n]*", "", f.read())
    if name == "sgmc_device.h":
      body = re.search(r"void wave_sync\(\) \{(.*?)\n\}", code, re.S)
      assert body and re.search(r'fence\(__ATOMIC_RELEASE, "wavefront"\);\s*'
                                r"__builtin_amdgcn_wave_barrier\(\);\s*"
                                r'__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "wavefront"\);',
                                body.group(1))
      code = code.replace(body.group(0), "")
    if "wave_barrier" in code:
      bare[name] = code.count("wave_barrier")
  assert not bare, bare
