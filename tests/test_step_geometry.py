"""CPU model of the whole-step patches (sbp_step.hpp step_plan, stencil_reach,
step2d_kernel): for many grid sizes and every order, the patches partition the
grid, every region fits a block's lanes and rows, and every point a stage's
stencil reads lies in the region the stage before it evaluated."""
import pytest

CLS, R, TAPS, ROWS = {2: 1, 4: 4, 6: 6}, {2: 1, 4: 2, 6: 3}, {2: 3, 4: 6, 6: 9}, {2: 24, 4: 24, 6: 32}
LANES, CUS = 64, 256


def reach(o, lo, hi, n):
    low, high = lo < CLS[o], hi > n - CLS[o]
    a, b = 0 if low else lo - R[o], n if high else hi + R[o]
    return min(n - TAPS[o], a) if high else a, max(TAPS[o], b) if low else b


def regions(o, lo, hi, n):
    """[loaded, stage 1, .., stage 4] of the patch [lo, hi) of a line of n points."""
    out = [(lo, hi)]
    for _ in range(4):
        out.insert(0, reach(o, *out[0], n))
    return out


def parts(n, length):
    return [(p, min(p + length, n)) for p in range(0, n, length)]


def fits(o, n, length, most):
    return all(hi - lo <= most for lo, hi in (regions(o, *p, n)[0] for p in parts(n, length)))


def plan(o, nx, ny):
    px = -(-nx // LANES)
    while not fits(o, nx, -(-nx // px), LANES):
        px += 1
    pw = -(-nx // px)
    px, best = -(-nx // pw), 0
    for ph in range(1, 9):
        if fits(o, ny, ph, ROWS[o]):
            best = ph
            if px * -(-ny // ph) <= CUS:
                break
    return pw, best


@pytest.mark.parametrize("order", [2, 4, 6])
def test_patches_cover_their_stencils(order):
    least = max(2 * CLS[order], TAPS[order])
    for n in list(range(least, 200)) + [257, 300, 385, 449, 513, 699, 1025]:
        pw, ph = plan(order, n, n)
        assert pw >= 1 and ph >= 1
        for length, most in ((pw, LANES), (ph, ROWS[order])):
            covered = 0
            for lo, hi in parts(n, length):
                assert lo == covered
                covered = hi
                e = regions(order, lo, hi, n)
                assert 0 <= e[0][0] and e[0][1] <= n and e[0][1] - e[0][0] <= most
                for st in range(1, 5):
                    for i in range(*e[st]):
                        if i < CLS[order]:
                            t = (0, TAPS[order])
                        elif i >= n - CLS[order]:
                            t = (n - TAPS[order], n)
                        else:
                            t = (i - R[order], i + R[order] + 1)
                        assert e[st - 1][0] <= t[0] and t[1] <= e[st - 1][1], (n, length, lo, st, i)
            assert covered == n
