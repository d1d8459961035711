"""The granular calls skip the media indices of single-medium tiles, whichever
passes the grid's fused calls run: media written between steps, and changes
of tiling, are followed."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd._lib import i32p, ptr
from test_quads import SPLIT, start

pytestmark = pytest.mark.gpu

PRIO = np.array([1000, 0, 20], np.int32)


def granular(s, n):
    for name in SPLIT:
        f = getattr(s.lib, "fdtd_" + name)
        assert (f(s.h, n) if "planewave" in name or "nodal" in name else f(s.h)) == 0, name


def fused(s, n):
    assert s.lib.fdtd_advance_e(s.h, n) == 0 and s.lib.fdtd_advance_h(s.h, n) == 0


@pytest.mark.parametrize("mode", ["exact", "fast"])
def test_granular_calls_follow_media_and_tilings(mode):
    pb = P.scatterer_problem(n=(67, 24, 22), L=((5, 4), (3, 4), (4, 3)), nsteps=40, disp=False)
    a, b = sf.Solver(pb, mode=mode), sf.Solver(pb, mode=mode)
    b.set_tiling(4, 8, 1)
    for s in (a, b):
        start(s, pb)
    n = 0
    for change in (None, "paint", (1, 5, 4), "paint", (2, 7, 1), (1, 64, 1), "paint", (4, 2, 4)):
        if change == "paint":
            for s in (a, b):
                assert s.lib.fdtd_media_paint_box(s.h, 10 + n, 30 + n, 4, 16, 2, 18, 2, 3, ptr(PRIO, i32p)) == 0
        elif change:
            a.set_tiling(*change)
        for _ in range(2):
            granular(a, n)
            fused(b, n)
            n += 1
        fused(a, n)
        granular(b, n)
        n += 1
        for c in range(6):
            assert np.array_equal(a.field(c).view(np.uint32), b.field(c).view(np.uint32)), (change, c)
    assert np.isfinite(a.field(0)).all() and np.abs(a.field(0)).max() > 0
