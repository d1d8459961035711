"""The observation launch (point probes and every frequency-domain box of a
grid in one kernel, the step counter moving once per recorded sequence):
boxes whose (point, frequency) pairs end at, before and after a block of 256
threads, several boxes of both kinds, and runs that mix the 16-step and the
one-step graphs."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P


def boxes(pairs):
    # one row of `pairs` points at one frequency, and a small H box beside it
    nx = pairs - 1
    return nx, [P.DftBox(0, (0, pairs - 1, 3, 3, 4, 4), (1, 1, 1), [1.1e9]),
                P.DftBox(1, (2, 4, 2, 5, 3, 3), (1, 1, 1), [0.7e9, 1.9e9, 2.3e9])]


@pytest.mark.gpu
@pytest.mark.parametrize("pairs,steps", [(255, 17), (256, 16), (257, 33), (300, 5)])
def test_sums_equal_direct_sums_of_probes(pairs, steps):
    nx, dfts = boxes(pairs)
    pb = P.scatterer_problem(n=(nx, 22, 20), nsteps=steps)
    pb.dfts = dfts
    pb.probes = [(0, pairs - 2, 3, 4), (1, pairs // 2, 3, 4), (5, 3, 4, 3), (3, 2, 2, 3)]
    s = sf.Solver(pb)
    s.run(steps)
    got, series = s.dft_sums(), s.probes().astype(np.float64)
    assert series.shape == (steps, 4)
    pi4 = float(np.float32(np.pi))
    t = np.concatenate([[0.0], np.cumsum(np.full(steps - 1, pb.dt))])
    # 64-bit sums of the same terms: the two differ by the rounding of at most
    # `steps` additions and of the phase factors, well under 1e-12 of the
    # largest partial sum
    for q, (box, comp, at) in enumerate([(0, 0, (0, 0, pairs - 2)), (0, 1, (0, 0, pairs // 2)),
                                         (1, 2, (0, 2, 1)), (1, 0, (0, 0, 0))]):
        for f, fr in enumerate(dfts[box].freqs):
            ph = pb.dt * np.exp(-1j * 2 * pi4 * float(fr) * (t + (pb.dt / 2 if box else 0.0)))
            want = np.sum(ph * series[:, q])
            scale = np.sum(np.abs(ph * series[:, q])) + 1e-300
            assert abs(got[box][at + (comp, f)] - want) <= 1e-12 * scale
    # call by call: the same samples and sums, bit for bit
    e = sf.Solver(pb)
    for _ in range(steps):
        e.step()
    assert np.array_equal(e.probes().view(np.uint32), series.astype(np.float32).view(np.uint32))
    for a, b in zip(e.dft_sums(), got):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
