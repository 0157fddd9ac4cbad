"""Values that lanes of one wave hand over through LDS are ordered for the
compiler too: a wave barrier is a scheduling barrier without memory semantics,
so every one in the sources stands between a release and an acquire fence."""
import os
import re

from problems_helper import ROOT

CSRC = os.path.join(ROOT, "hpc-reading-course_amd", "csrc")


def test_wave_barriers_stand_between_fences():
    found = 0
    for f in sorted(os.listdir(CSRC)):
        text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, f)).read())
        calls = [s.strip() for s in re.split(r"[;{}]", text) if s.strip()]
        for k, call in enumerate(calls):
            if "__builtin_amdgcn_wave_barrier()" not in call:
                continue
            found += 1
            assert calls[k - 1] == '__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront")', f
            assert calls[k + 1] == '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront")', f
    assert found
