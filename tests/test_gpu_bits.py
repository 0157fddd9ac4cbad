"""Every schedule forms the same bits in every precision: whole steps (patches,
marched), two stages per launch and one, from the same state; and lines of
several tiles whatever their launches' cuts, the compensation included.

Bar: equality.  FP64 sums are written in one order, FP32 multiply-adds are
written out and never left to contraction, so nothing may differ.
"""
import importlib

import numpy as np
import pytest

from problems_helper import P
from test_gpu_line import problem as line_problem
from test_gpu_step import problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    return importlib.import_module("hpc-reading-course_amd.capi")


@pytest.mark.parametrize("prec", [P.FP64, P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("kind,order,nx,ny,bc,whole", [
    ("unit", 2, 23, 31, P.BC_WALL, "patches"), ("arrays", 4, 65, 66, P.BC_WALL, "patches"),
    ("ref", 4, 130, 97, P.BC_FREE_SURFACE, "patches"), ("ref", 6, 65, 120, P.BC_DEFAULT, "patches"),
    ("arrays", 6, 97, 65, P.BC_FREE_SURFACE_REF, "patches"), ("adv", 2, 40, 300, P.BC_DEFAULT, "patches"),
    ("swirl", 4, 129, 66, P.BC_DEFAULT, "patches"), ("unit", 2, 600, 555, P.BC_WALL, "march"),
    ("unit", 4, 555, 600, P.BC_FREE_SURFACE, "march"), ("arrays", 4, 501, 600, P.BC_WALL, "march"),
    ("arrays", 6, 601, 505, P.BC_WALL, "march"), ("unit", 6, 505, 601, P.BC_DEFAULT, "march"),
    ("adv", 4, 600, 501, P.BC_DEFAULT, "march"), ("swirl", 6, 520, 601, P.BC_DEFAULT, "march")])
def test_schedules_agree_to_the_bit(capi, kind, order, nx, ny, bc, whole, prec):
    print("bits", kind, order, nx, ny, bc, prec, flush=True)
    spec, v, _ = problem(kind, order, nx, ny, bc, prec)
    dt = 0.2 / max(spec.hix, spec.hiy)
    out = {}
    with capi.Context(spec) as ctx:
        for choice in (None, False, True):
            if choice is not None:
                ctx.set_fused(choice)
            ctx.set_state(v)
            ctx.step(0.3, dt, 19)  # a replayed graph of 16 where there is no forcing, then 3 launches
            out[ctx.schedule] = ctx.get_state()
    assert set(out) == {whole, "stages", "pairs"}
    assert np.any(out["stages"]) and np.all(np.isfinite(out["stages"]))
    for name, o in out.items():
        assert np.array_equal(o, out["stages"]), name


@pytest.mark.parametrize("prec", [P.FP64, P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("kind,order,n,steps", [("refl", 6, 1001, 11), ("adv", 4, 3 * 112 + 1, 15), ("var", 2, 401, 45),
                                                ("refl", 4, 256 * 112 + 1, 13)])
def test_line_launch_cuts_do_not_show(capi, kind, order, n, steps, prec):
    """One call of many steps (4 to 20 per launch) against a call per step: the
    state and its compensation trade arrays at other times."""
    print("line cuts", kind, order, n, steps, prec, flush=True)
    spec, v, dt = line_problem(kind, n, order, prec)
    with capi.Context(spec) as ctx:
        ctx.set_state(v)
        ctx.step(0.0, dt, steps)
        many = ctx.get_state()
        ctx.set_state(v)
        for _ in range(steps):
            ctx.step(0.0, dt, 1)
        assert np.array_equal(ctx.get_state(), many)
    if prec == P.FP32_KAHAN:  # the compensation is there: it changes the sum
        with capi.Context(spec.with_(precision=P.FP32)) as ctx:
            assert not np.array_equal(ctx.rk4_advance(v, 0.0, dt, steps), many)
