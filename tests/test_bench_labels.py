"""The benchmark names the kernel that a context's schedule runs."""
import importlib

import pytest

import problems_helper  # noqa: F401  (puts the repository on sys.path)

bench = importlib.import_module("bench")
capi = importlib.import_module("hpc-reading-course_amd.capi")


@pytest.mark.parametrize("sched,slots", [("stages", {1: "stage2d", 2: "stage2d", 3: "stage2d", 4: "stage2d"}),
                                         ("pairs", {1: "pair2d", 3: "pair2d"}), ("patches", {1: "step2d"}),
                                         ("march", {1: "march2d"}), ("line", {1: "line"})])
def test_kernel_of_every_schedule(sched, slots):
    assert set(bench.SCHEDULE) == set(capi.SCHEDULES)
    names = bench.kernel_names(sched)
    assert {k: n.split("_kernel")[0] for k, n in names.items() if n != "(no launch)"} == slots
