"""Marched RK4 steps (march2d_kernel) against one launch per stage, at the
edges of strips and segments: the smallest grids that march, one strip and one
column more, ribbons, ragged sizes.

Bars: FP64 bit-identical (same arithmetic per point) and within 1e-12 of the
CPU oracle; FP32 and FP32+Kahan within 2e-6 of one launch per stage, the bar
the other schedules have.
"""
import importlib

import numpy as np
import pytest

from problems_helper import P
from test_gpu_step import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [P.FP64, P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("kind,order,nx,ny,bc", [
    ("unit", 2, 256, 267, P.BC_WALL), ("arrays", 2, 504, 141, P.BC_FREE_SURFACE), ("adv", 2, 257, 601, P.BC_DEFAULT),
    ("unit", 4, 261, 570, P.BC_DEFAULT), ("arrays", 4, 500, 301, P.BC_WALL), ("swirl", 4, 501, 389, P.BC_DEFAULT),
    ("unit", 4, 131, 1201, P.BC_FREE_SURFACE), ("adv", 4, 1201, 129, P.BC_DEFAULT), ("unit", 4, 1025, 515, P.BC_WALL),
    ("unit", 6, 262, 580, P.BC_DEFAULT), ("arrays", 6, 495, 337, P.BC_FREE_SURFACE), ("swirl", 6, 494, 401, P.BC_DEFAULT),
    ("arrays", 6, 37, 13300, P.BC_WALL)])
def test_marched_steps_match_stage_launches(orc, kind, order, nx, ny, bc, prec):
    capi = importlib.import_module("hpc-reading-course_amd.capi")
    print("marched step", kind, order, nx, ny, bc, prec, flush=True)
    spec, v, _ = problem(kind, order, nx, ny, bc, prec)
    dt = 0.2 / max(spec.hix, spec.hiy)  # stable on ribbons too
    with capi.Context(spec) as ctx:
        ctx.set_state(v)
        ctx.step(0.0, dt, 19)  # a replayed graph of 16, then 3 launches
        got = ctx.get_state()
        ms = ctx.time_stages(dt, 1)
        assert ms[0] > 0 and not ms[1:].any()
    with capi.Context(spec) as ctx:
        ctx.set_fused(False)
        ctx.set_state(v)
        ctx.step(0.0, dt, 19)
        want = ctx.get_state()
    if prec == P.FP64:
        assert np.array_equal(got, want)
        ref = orc.rk4(spec, v, 0.0, dt, 5)
        with capi.Context(spec) as ctx:
            ctx.set_state(v)
            ctx.step(0.0, dt, 5)
            got = ctx.get_state()
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
    else:
        assert np.max(np.abs(got - want)) <= 2e-6 * np.max(np.abs(want))
