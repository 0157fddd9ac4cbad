"""Tile heights of one launch per stage: remainder rows, one row, one tile.
Every height gives the same bits, which are the default schedule's.

Bars: FP64 equal to the bit, FP32 and FP32+Kahan too (multiply-adds are fused
where the source says so, the same way in every kernel).
"""
import importlib

import numpy as np
import pytest

from problems_helper import P
from test_gpu_step import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [P.FP64, P.FP32, P.FP32_KAHAN])
@pytest.mark.parametrize("kind,order,nx,ny", [("unit", 6, 300, 300), ("arrays", 4, 261, 97), ("ref", 2, 130, 259),
                                              ("swirl", 4, 513, 70)])
def test_tile_rows_of_stage_launches(kind, order, nx, ny, prec):
    capi = importlib.import_module("hpc-reading-course_amd.capi")
    print("tile rows", kind, order, nx, ny, prec, flush=True)
    spec, v, dt = problem(kind, order, nx, ny, P.BC_DEFAULT, prec)
    with capi.Context(spec) as ctx:
        assert ctx.schedule in ("patches", "march")
        want = ctx.rk4_advance(v, 0.1, dt, 3)
        ctx.set_fused(False)
        for rows in (1, 7, 16, 64, 300):
            ctx.set_tile_rows(rows)
            assert ctx.schedule == "stages"
            assert np.array_equal(ctx.rk4_advance(v, 0.1, dt, 3), want), rows
