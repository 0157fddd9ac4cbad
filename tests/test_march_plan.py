"""march_plan itself (sbp_step.hpp, compiled for the host): where a CU holds one
block, patches of the frame that have to wait for the strips' blocks cost a
second block's time, and a plan lets them only if that saves more rows."""
import os
import subprocess

import numpy as np
import pytest

from problems_helper import ROOT
from test_march_geometry import CUS, DEPTH, ceil, plan

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plans") / "plans")
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "--offload-host-only", "-I",
                    os.path.join(ROOT, "hpc-reading-course_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "plans.hip"), "-o", exe], check=True)

    def run(grids):
        r = subprocess.run([exe], input="\n".join("%d %d %d %d" % g for g in grids), stdout=subprocess.PIPE, text=True,
                           check=True)
        return [tuple(int(v) for v in l.split()) for l in r.stdout.splitlines()]

    return run


def sizes(order, count):
    rng = np.random.default_rng(order)
    lo = 2 * DEPTH[order] + 1
    out = [(1395, 129), (1133, 132), (129, 1395), (178, 1145), (500, 800), (1025, 1025), (4097, 4097), (lo, lo), (lo, 5000)]
    while len(out) < count:
        n = np.exp(rng.uniform(np.log(lo + 1), np.log(5000), 2)).astype(int)
        out.append(tuple(int(v) for v in n))
    return out


@pytest.mark.parametrize("order", [2, 4, 6])
def test_one_block_per_cu(plans, order):
    grids = sizes(order, 400)
    waiting = 0
    for (nx, ny), (ok, strips, segs, rows, nf) in zip(grids, plans([(order, nx, ny, 1) for nx, ny in grids])):
        h = ny - 2 * DEPTH[order]
        assert ok and segs == ceil(h, rows) and strips == ceil(nx - 2 * DEPTH[order], 256 - 4 * order)
        within = CUS - nf
        if strips * segs + nf > CUS and within >= strips:
            waiting += 1  # all blocks at once would run more rows, in whole groups, than a wait costs
            group = order + 1
            assert ceil(ceil(h, within // strips), group) * group > ceil(rows, group) * group + 3 * order, (nx, ny)
    assert 0 < waiting < len(grids) // 2


@pytest.mark.parametrize("order", [2, 4, 6])
def test_several_blocks_per_cu(plans, order):
    grids = sizes(order, 100)
    for resident in (2, 4, 7):
        for (nx, ny), got in zip(grids, plans([(order, nx, ny, resident) for nx, ny in grids])):
            px = (got[4] - 2 * ceil(ny - 2 * DEPTH[order], 64 - 4 * order)) // 2
            assert got[0] and got[1:4] == plan(order, nx, ny, px, resident)
