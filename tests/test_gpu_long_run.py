"""Long FP32 and FP32+Kahan runs of the variable-material order-6 workload (rho,
K from 8 seeded Gaussians in [0.5, 2], wall SATs, Gaussian pulse, CFL 0.25)
against the FP64 oracle, by every schedule: 2000 steps at 257^2 in one launch per
stage and in patches, 400 steps marched at 505^2 (the schedule of the 4097^2
run), with the two-stage schedule beside it.

Bar: 2e-5 relative max norm, the FP32 bar of the other paths.
"""
import importlib
import os

import numpy as np
import pytest

from problems_helper import P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("n,steps,schedules", [(257, 2000, ("patches", "stages")), (505, 400, ("march", "pairs"))])
def test_reflection_workload_by_schedule(orc, prec, n, steps, schedules):
    capi = importlib.import_module("hpc-reading-course_amd.capi")
    spec, v0, dt = P.baseline_reflection(n, precision=prec)
    ref = orc.rk4(spec.with_(precision=P.FP64), v0, 0.0, dt, steps, threads=min(16, os.cpu_count() or 1))
    for schedule in schedules:
        with capi.Context(spec) as ctx:
            if schedule in ("stages", "pairs"):
                ctx.set_fused(schedule == "pairs")
            assert ctx.schedule == schedule
            got = ctx.rk4_advance(v0, 0.0, dt, steps)
        err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
        print("reflection workload", n, prec, schedule, "%.3e" % err, flush=True)
        assert err <= 2e-5
