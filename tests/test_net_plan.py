"""The cut of the corrector's images into chunks of rows (sbp_corr_plan.hpp): the
split of the least modelled time among all even ones, found in a time that does
not grow with the image; it is asked for at every launch."""
import os
import subprocess

import numpy as np
import pytest

from problems_helper import ROOT

CUS, OUT, HALO, MOST = 256, 58, 9, 32


def ceil(a, b):
    return -(-a // b)


def best_rows(nb, H, W):
    """Every number of chunks that keeps them within MOST rows, the first of the least."""
    strips = nb * ceil(W, OUT)
    least, rows = None, None
    for n in range(ceil(H, MOST), H + 1):
        r = ceil(H, n)
        cost = ceil(r + HALO, 6) * 6 * max(0.55, 0.43 * ceil(strips * ceil(H, r), CUS))
        if least is None or cost < least:
            least, rows = cost, r
    return rows


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "net_plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "hpc-reading-course_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "net_plan.cpp"), "-o", exe], check=True)

    def run(cases, timeout=60):
        r = subprocess.run([exe], input="\n".join("%d %d %d" % c for c in cases), stdout=subprocess.PIPE, text=True,
                           check=True, timeout=timeout)
        return [tuple(int(v) for v in l.split()) for l in r.stdout.splitlines()]

    return run


def test_chunks_are_the_least_of_all_even_splits(plans):
    rng = np.random.default_rng(0)
    cases = [(1, 3, 3), (1, 257, 257), (16, 257, 257), (4, 257, 257), (1, 33, 58), (3, 32, 59), (1, 4097, 4097), (256, 65, 65)]
    cases += [(int(rng.integers(1, 40)), int(np.exp(rng.uniform(1.1, 6.5))), int(np.exp(rng.uniform(1.1, 7)))) for _ in range(400)]
    for (nb, H, W), (rows, blocks, most) in zip(cases, plans(cases)):
        assert rows == best_rows(nb, H, W), (nb, H, W)
        assert blocks == ceil(W, OUT) * ceil(H, rows) <= most


def test_tall_images_cost_no_search(plans):
    """A million calls on images of 2^26 rows, one of which was 67 million trials."""
    out = plans([(1, 1 << 26, 3)] * 1000000, timeout=30)
    assert len(out) == 1000000 and all(1 <= r <= MOST for r, _, _ in out[:3])
