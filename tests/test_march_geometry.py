"""CPU model of marched steps (sbp_step.hpp march_plan, sbp_march.hpp): for
many grid sizes and every order, strips, segments and frame patches write every
point exactly once, all reads stay in the grid, and no strip or side patch
evaluates a closure point of the operator where it uses the interior stencil."""
import numpy as np
import pytest

from test_step_geometry import CLS, R, regions

THREADS, LANES, CUS = 256, 64, 256
DEPTH = {2: 4, 4: 10, 6: 15}


def ceil(a, b):
    return -(-a // b)


def plan(o, nx, ny, px, resident):
    w, h = nx - 2 * DEPTH[o], ny - 2 * DEPTH[o]
    cols = THREADS - 4 * o
    strips = ceil(w, cols)
    nf = 2 * px + 2 * ceil(h, LANES - 4 * o)
    best = None
    for per in range(1, resident + 1):
        slots = CUS * per
        blocks = slots - nf if 4 * nf <= slots else slots
        rows = ceil(h, max(1, blocks // strips))
        cost = (rows + 4 * o) * (4 + per)
        if best is None or cost < best[0]:
            best = cost, rows
    return strips, ceil(h, best[1]), best[1]


@pytest.mark.parametrize("resident", [1, 2, 4, 7])
@pytest.mark.parametrize("order", [2, 4, 6])
def test_strips_and_frame_partition_the_grid(order, resident):
    D, r, cls = DEPTH[order], R[order], CLS[order]
    assert D == cls + 3 * r
    cols, side = THREADS - 4 * order, LANES - 4 * order
    assert 4 * order == 8 * r
    rng = np.random.default_rng(order)
    sizes = [(2 * D + 1, 2 * D + 1), (2 * D + cols, 401), (2 * D + cols + 1, 389), (1025, 1025), (130, 1201)]
    sizes += [tuple(int(n) for n in rng.integers(2 * D + 1, 900, 2)) for _ in range(8)]
    for nx, ny in sizes:
        pw = 36  # any width whose regions fit the lanes
        px = ceil(nx, pw)
        strips, segs, rows = plan(order, nx, ny, px, resident)
        seen = np.zeros((ny, nx), dtype=np.int32)
        for s in range(strips):
            i = D + s * cols - 4 * r + np.arange(THREADS)
            assert i[0] >= 0  # loads are clamped to nx - 1 only
            t = np.arange(THREADS)
            out = i[(t >= 4 * r) & (t < THREADS - 4 * r) & (i < nx - D)]
            assert len(out) and out[0] - 3 * r >= cls and out[-1] + 3 * r < nx - cls
            for g in range(segs):
                j0, j1 = D + g * rows, min(D + (g + 1) * rows, ny - D)
                assert j1 > j0 and j0 - 4 * r >= 0
                seen[j0:j1, out] += 1
        loaded = ceil(D + 4 * r, THREADS // 64) * (THREADS // 64)
        for lo, hi in ((0, D), (ny - D, ny)):
            assert np.ptp(regions(order, lo, hi, ny)[0]) <= loaded
            for p in range(px):
                i0, i1 = p * pw, min((p + 1) * pw, nx)
                assert np.ptp(regions(order, i0, i1, nx)[0]) <= LANES
                seen[lo:hi, i0:i1] += 1
        for lo, hi in ((0, D), (nx - D, nx)):
            assert np.ptp(regions(order, lo, hi, nx)[0]) <= loaded
            for p in range(ceil(ny - 2 * D, side)):
                j0, j1 = D + p * side, min(D + (p + 1) * side, ny - D)
                e = regions(order, j0, j1, ny)
                assert np.ptp(e[0]) <= LANES and e[0][0] >= 0 and e[1][0] >= cls and e[1][1] <= ny - cls
                seen[j0:j1, lo:hi] += 1
        assert (seen == 1).all(), (nx, ny)
