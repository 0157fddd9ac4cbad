"""CPU model of the patches of one-launch RKF4(5) attempts (sbp_step.hpp
patch_plan, sbp_rkf.hpp): wherever a cut exists, its patches partition the
grid, every six-stage region fits a block's lanes and rows, and every point a
stage reads was evaluated by the stage before it."""
import pytest

from test_step_geometry import CLS, CUS, LANES, R, TAPS, parts, reach

ROWS = {2: 32, 4: 32, 6: 40}


def regions(o, lo, hi, n):
    out = [(lo, hi)]
    for _ in range(6):
        out.insert(0, reach(o, *out[0], n))
    return out


def fits(o, n, length, most):
    return all(hi - lo <= most for lo, hi in (regions(o, *p, n)[0] for p in parts(n, length)))


def plan(o, nx, ny):
    px = -(-nx // LANES)
    while not fits(o, nx, -(-nx // px), LANES):
        if -(-nx // px) == 1:
            return None
        px += 1
    pw = -(-nx // px)
    px, best = -(-nx // pw), 0
    for ph in range(1, 21):
        if fits(o, ny, ph, ROWS[o]):
            best = ph
            if px * -(-ny // ph) <= CUS:
                break
    return (pw, best) if best else None


@pytest.mark.parametrize("order", [2, 4, 6])
def test_patches_cover_their_stencils(order):
    least, planned = max(2 * CLS[order], TAPS[order]), 0
    for n in list(range(least, 180)) + [257, 303, 401, 701, 1100]:
        cut = plan(order, n, n)
        if not cut:
            continue
        planned += 1
        for length, most in ((cut[0], LANES), (cut[1], ROWS[order])):
            covered = 0
            for lo, hi in parts(n, length):
                assert lo == covered
                covered = hi
                e = regions(order, lo, hi, n)
                assert 0 <= e[0][0] and e[0][1] <= n and e[0][1] - e[0][0] <= most
                for st in range(1, 7):
                    for i in range(*e[st]):
                        if i < CLS[order]:
                            t = (0, TAPS[order])
                        elif i >= n - CLS[order]:
                            t = (n - TAPS[order], n)
                        else:
                            t = (i - R[order], i + R[order] + 1)
                        assert e[st - 1][0] <= t[0] and t[1] <= e[st - 1][1], (n, length, lo, st, i)
            assert covered == n
    assert planned > 100
