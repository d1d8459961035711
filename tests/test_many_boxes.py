"""Frequency-domain boxes of a grid that share a launch (each starts on a block
of its own): sums equal those of the same box alone, for boxes whose (point,
frequency) pairs end around a block, alone and in a batch; large boxes in the
recorded steps against the call-by-call ones."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd.batch import Batch
from test_quads import start

pytestmark = pytest.mark.gpu


def grid(dfts, n=(300, 12, 14), storage="fp32"):
    pb = P.scatterer_problem(n=n, L=((4, 4), (3, 2), (2, 3)), nsteps=40, disp=False)
    pb.dfts = dfts
    s = sf.Solver(pb, storage=storage)
    start(s, pb)
    return s


def row(kind, pairs, nf=1):
    return P.DftBox(kind, (1, pairs // nf, 3, 3, 4, 4), (1, 1, 1), list(np.linspace(0.5e9, 2e9, nf)))


def equal(a, b):
    return np.abs(a).max() > 0 and np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
def test_boxes_side_by_side(storage):
    boxes = [row(1, 1), row(0, 255), row(0, 256), row(1, 257), row(0, 3, 3), row(1, 64), row(0, 65),
             row(1, 510, 2), row(0, 1), P.DftBox(0, (2, 290, 1, 9, 2, 9), (3, 2, 2), [1.1e9, 0.9e9])]
    steps = 19
    want = []
    for b in boxes:
        s = grid([b], storage=storage)
        s.run(steps)
        want.append(s.dft_sums()[0])
        s.close()
    s = grid(boxes, storage=storage)
    s.run(steps)
    for k, (g, w) in enumerate(zip(s.dft_sums(), want)):
        assert equal(g, w), k
    batch = Batch()
    sol = [grid(boxes[k:], storage=storage) for k in (0, 5)]
    for q in sol:
        batch.admit(q)
    batch.step(steps)
    for q, k in zip(sol, (0, 5)):
        for g, w in zip(q.dft_sums(), want[k:]):
            assert equal(g, w), k
    batch.close()


@pytest.mark.parametrize("rows", [1, 4])
def test_large_boxes_recorded(rows):
    n, box = (76, 76, 76), (1, 70, 1, 70, 1, 70)
    dfts = [P.DftBox(1, box, (1, 1, 1), [0.7e9]), P.DftBox(0, box, (1, 1, 1), [1.1e9, 1.9e9])]
    a, b = grid(dfts, n), grid(dfts, n)
    a.set_tiling(rows, 1, 4)
    a.run(18)
    for _ in range(18):
        b.step()
    assert np.array_equal(a.probes().view(np.uint32), b.probes().view(np.uint32))
    for x, y in zip(a.dft_sums(), b.dft_sums()):
        assert equal(x, y)
