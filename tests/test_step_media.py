"""Media written between one-launch steps of a grid with poles: its pole state
starts again, the stored previous field among it, as in the two passes."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd._lib import i32p, ptr
from semba_fdtd_amd.batch import Batch
from test_quads import start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["run", "batch"])
@pytest.mark.parametrize("mode", ["exact", "fast"])
def test_media_between_one_launch_steps(mode, how):
    pb = P.scatterer_problem(n=(46, 35, 27), L=((3, 4), (2, 3), (3, 2)), nsteps=60, mdisp=True)
    prio = np.array([1000] + [0] * pb.nmedia, np.int32)
    prio[2] = 50
    a, b = sf.Solver(pb, mode=mode), sf.Solver(pb, mode=mode)
    a.set_step_mode(8, 9)
    batch = Batch(step_rows=8, step_zchunk=9)
    for s in (a, b):
        start(s, pb)

    def go(n):
        if how == "run":
            a.run(n)
        else:
            slot = batch.admit(a)
            batch.step(n)
            batch.retire(slot)
        b.run(n)

    go(12)
    for at in (20, 10):
        for s in (a, b):
            assert s.lib.fdtd_media_paint_box(s.h, at, at + 8, 10, 16, 8, 15, 2, len(prio), ptr(prio, i32p)) == 0
        go(14)
        for c in range(6):
            x, y = a.field(c), b.field(c)
            assert np.abs(y).max() > 0 and np.array_equal(x.view(np.uint32), y.view(np.uint32)), (at, c)
    batch.close()
