"""Plane-wave boxes that reach the grid's edge, whose faces act on cells outside
their components' sweeps, with one-launch steps asked for: the oracle's bits,
alone and in a batch."""
import numpy as np
import pytest

import oracle
import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd.batch import Batch
from test_inline_sources import STEPS, wave

pytestmark = pytest.mark.gpu

BOXES = {"all": (0, 40, 0, 26, 0, 24), "low z": (5, 30, 5, 20, 0, 20), "high": (5, 40, 5, 26, 5, 24),
         "inside": (1, 39, 1, 25, 1, 23)}


def problem(box):
    pb = P.scatterer_problem(n=(40, 26, 24), L=((0, 0),) * 3, nsteps=STEPS, disp=False)
    pb.planewaves = [wave(pb, box)]
    return pb


def check(s, ref):
    for c in range(6):
        assert np.array_equal(s.field(c).view(np.uint32), ref.fields[c].view(np.uint32)), c


@pytest.mark.parametrize("name", list(BOXES))
def test_boxes_on_the_edge(name):
    pb = problem(BOXES[name])
    ref = oracle.Oracle(pb)
    ref.run(STEPS)
    s = sf.Solver(pb, mode="exact")
    s.set_step_mode(8, 8)
    s.run(STEPS)
    check(s, ref)
    both = [sf.Solver(pb, mode="exact"), sf.Solver(problem(BOXES["inside"]), mode="exact")]
    b = Batch(step_rows=8, step_zchunk=8)
    for q in both:
        b.admit(q)
    b.step(STEPS)
    check(both[0], ref)
    b.close()
