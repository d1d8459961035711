"""Which work a batch launches: its own one-launch steps observe and nothing
more."""
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
