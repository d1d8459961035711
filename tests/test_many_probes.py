"""Probes of a grid spread over blocks of a face pass where one block's threads
do not hold them: every sample of runs on the 16-step, the 4-step and the
one-step graph equals the call-by-call one."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from test_quads import start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiling", [None, (2, 3, 4), (4, 4, 4), (2, 4, 1)])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 128, 257, 1500])
def test_every_probe_sampled(count, tiling):
    pb = P.scatterer_problem(n=(30, 22, 20), nsteps=40)
    rng = np.random.default_rng(count)
    pb.probes = [(int(rng.integers(0, 6)), int(rng.integers(0, 30)), int(rng.integers(0, 22)),
                  int(rng.integers(0, 20))) for _ in range(count)]
    pb.dfts = [P.DftBox(1, (2, 20, 3, 9, 3, 6), (3, 1, 1), [0.7e9, 1.9e9]),
               P.DftBox(0, (1, 25, 2, 9, 3, 3), (2, 2, 1), [1.1e9])]
    a, b = sf.Solver(pb), sf.Solver(pb)
    for s in (a, b):
        if tiling:
            s.set_tiling(*tiling)
        start(s, pb)
    a.run(18)
    a.set_graph_steps(4)
    a.run(7)
    for _ in range(25):
        b.step()
    want = b.probes()
    assert want.shape == (25, count) and np.abs(want).min(axis=0).max() > 0
    assert np.array_equal(a.probes().view(np.uint32), want.view(np.uint32))
    for x, y in zip(a.dft_sums(), b.dft_sums()):
        assert np.abs(x).max() > 0 and np.array_equal(x.view(np.uint64), y.view(np.uint64))
