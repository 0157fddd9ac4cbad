"""Whole-step 1D kernel (line_kernel) at the edges of its tiles: one block,
two blocks, a last block of one point, the changes of block size, step counts
around the steps of one launch.

Bars: FP64 bit-identical to the CPU oracle (same operation order, no FMA
contraction).  FP32 and FP32+Kahan within 2e-5 of the FP64 oracle (the FP32
bar of the other paths), and resident state read back in the middle.
"""
import importlib

import numpy as np
import pytest

from problems_helper import P

pytestmark = pytest.mark.gpu


def problem(kind, n, order, prec=P.FP64):
    if kind == "var":
        spec, v = P.adv1d_var(n, order, precision=prec)
    else:
        spec, v = (P.reflection if kind == "refl" else P.adv1d)(n, order, precision=prec)
    return spec, v + 0.05 * np.random.default_rng(n).standard_normal(v.size), P.dt_from_cfl(spec, 0.2)


# tiles: order 2 96 points (20 steps a launch), order 4 112 (6), order 6 96 (4)
@pytest.mark.parametrize("kind,order,n,steps", [
    ("adv", 2, 3, 7), ("refl", 4, 8, 30), ("adv", 6, 12, 1025), ("refl", 2, 255, 41), ("adv", 4, 256, 13),
    ("refl", 6, 257, 9), ("adv", 4, 2 * 112 + 1, 5), ("refl", 4, 3 * 112 + 1, 6), ("var", 2, 4 * 96 + 1, 21),
    ("refl", 6, 3 * 96 + 5, 4), ("var", 6, 1025, 11), ("adv", 4, 256 * 112 + 1, 19), ("refl", 6, 256 * 96 + 1, 17),
    ("adv", 2, 256 * 704 + 1, 23)])
def test_line_fp64_bit_identical(orc, kind, order, n, steps):
    capi = importlib.import_module("hpc-reading-course_amd.capi")
    print("line", kind, order, n, steps, flush=True)
    spec, v, dt = problem(kind, n, order)
    with capi.Context(spec) as ctx:
        ctx.set_state(v)
        ctx.step(0.0, dt, steps // 2)
        mid = ctx.get_state()
        ctx.step(0.0, dt, steps - steps // 2)
        got = ctx.get_state()
    assert np.array_equal(mid, orc.rk4(spec, v, 0.0, dt, steps // 2))
    assert np.array_equal(got, orc.rk4(spec, v, 0.0, dt, steps))


@pytest.mark.parametrize("prec", [P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("kind,order,n", [("refl", 4, 200), ("adv", 6, 500), ("refl", 2, 30001), ("var", 4, 113)])
def test_line_fp32(orc, kind, order, n, prec):
    capi = importlib.import_module("hpc-reading-course_amd.capi")
    print("line fp32", kind, order, n, prec, flush=True)
    spec, v, dt = problem(kind, n, order, prec)
    with capi.Context(spec) as ctx:
        got = ctx.rk4_advance(v, 0.0, dt, 33)
    ref = orc.rk4(spec.with_(precision=P.FP64), v, 0.0, dt, 33)
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref))
