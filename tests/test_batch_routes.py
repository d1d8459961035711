"""Which work a batch launches: its one-launch steps observe and nothing more,
its passes run the tiling they are asked for."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd.batch import Batch

pytestmark = pytest.mark.gpu


def batch_plan(b):
    """[four cells per lane, tiles of the passes, observation blocks of a
    two-pass step, of a one-launch step]"""
    out = np.zeros(4, np.int32)
    assert b.lib.sfd_batch_plan(b.b, out.ctypes) == 0
    return out


def test_one_launch_steps_compute_no_two_pass_terms():
    """The plane wave's next terms ride with the observation of a two-pass
    step; a one-launch step has a launch of its own for its incident field."""
    pb = P.open_scatterer_problem(n=32, L=5, radius=4, nsteps=40)
    pb.probes = []
    sol = [sf.Solver(pb) for _ in range(3)]
    b = Batch(step_rows=8)
    for s in sol:
        b.admit(s)
    b.step(5)
    plan = batch_plan(b)
    assert plan[2] > 0 and plan[3] == 0
    b.close()


def test_asked_tilings_are_run():
    """Left alone a batch chooses its passes; rows, planes and cells per lane
    asked for are the ones that run, whoever asks."""
    pb = P.scatterer_problem(n=(60, 30, 40), L=((0, 0),) * 3, nsteps=30, disp=False)
    flat = -(-61 * 31 // 128) * -(-41 // 8)         # runs of 2 rows, 8 planes
    quad = -(-16 * 31 // 128) * -(-41 // 8)
    for b, want in ((Batch(), (1, None)), (Batch(rows=2, zchunk=8, xcells=1), (0, flat)),
                    (Batch(rows=2, zchunk=8), (0, flat)), (Batch(xcells=1), (0, None)),
                    (Batch(rows=2, zchunk=8, xcells=4), (1, quad))):
        s = sf.Solver(pb)
        slot = b.admit(s)
        b.step(2)
        plan = batch_plan(b)
        assert plan[0] == want[0] and want[1] in (None, plan[1])
        b.set_tiling(2, 8, 64, 1)
        b.step(2)
        assert list(batch_plan(b)[:2]) == [0, flat]
        b.retire(slot)
        b.close()
        s.close()
