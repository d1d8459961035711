"""Sources inside the one-cell face passes (TF/SF faces by index masks, nodal
cells per tile) against the separate source launches that follow the four-cell
passes: the same bits, for every kind of source the passes take and for those
they leave to the separate launches."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P

STEPS = 40


def wave(pb, box, p=(0.0, 0.0, 1.0), e=(1.0, 0.0, 0.0)):
    q = np.arange(STEPS + 5)
    ev = (np.sin(q / 5.0) * (1 - np.exp(-q / 4.0))).astype(np.float32)
    return P.PlaneWave(box, [p], [e], ev, float(np.float32(pb.dt)))


def nodal(pb, comp, hard, box, amp):
    ev = P.gaussian_table(pb.dt, STEPS + 4, 6.0, 10.0)
    return P.NodalSource(comp, hard, box, amp, ev, float(np.float32(pb.dt)))


def build(kind, nx=70):
    open_ = dict(n=(nx, 26, 24), L=((4, 5), (3, 4), (5, 3)), nsteps=STEPS)
    pb = P.scatterer_problem(**open_, disp=kind != "plain", soft=True)
    inner = (6, nx - 7, 5, 20, 7, 19)
    if kind in ("plain", "poles"):
        pb.planewaves = [wave(pb, inner)]
    elif kind == "oblique":
        pb.planewaves = [wave(pb, inner, (0.48, 0.64, 0.6), (0.8, -0.6, 0.0))]
    elif kind == "pole_face":        # a face through the pole medium: separate launches
        pb.planewaves = [wave(pb, (6, nx - 7, 5, 20, 8, 19))]
    elif kind == "three_waves":      # 36 faces per half, more than the masks hold
        pb.planewaves = [wave(pb, (6 + d, nx - 7 - d, 5 + d, 20 - d, 7 + d, 19 - d)) for d in range(3)]
    elif kind == "two_waves":
        pb.planewaves = [wave(pb, inner), wave(pb, (8, nx - 7, 5, 18, 7, 17), (0.0, 0.6, 0.8), (1.0, 0.0, 0.0))]
    elif kind == "edge":             # no CPML, the box on the grid's edge: faces outside the sweep
        pb = P.scatterer_problem(n=(nx, 26, 24), L=((0, 0),) * 3, nsteps=STEPS, disp=False)
        pb.planewaves = [wave(pb, (0, nx, 0, 26, 0, 24))]
    elif kind == "nodal_box":        # many cells over many tiles, on the wave's faces too
        pb.planewaves = [wave(pb, inner)]
        pb.nodal = [nodal(pb, P.EX, False, (10, nx - 9, 5, 20, 15, 16), 2.0),
                    nodal(pb, P.HZ, False, (9, 40, 6, 12, 14, 15), 0.01)]
    elif kind == "nodal_shared":     # cells written twice: in order, hard before soft
        pb.nodal = [nodal(pb, P.EZ, False, (20, 30, 8, 12, 12, 14), 2.0),
                    nodal(pb, P.EZ, True, (25, 40, 10, 16, 13, 15), 0.5),
                    nodal(pb, P.HY, True, (25, 27, 10, 11, 13, 15), 0.02)]
    return pb


KINDS = ["plain", "poles", "oblique", "pole_face", "three_waves", "two_waves", "edge", "nodal_box",
         "nodal_shared"]


def run(pb, mode, storage, xcells, rows=2, zchunk=4):
    s = sf.Solver(pb, mode=mode, storage=storage)
    s.set_tiling(rows, zchunk, xcells)
    s.run(STEPS - 1)
    s.step() if storage == "fp32" else s.run(1)
    return s.probes(), [s.field(c) for c in range(6)]


@pytest.mark.gpu
@pytest.mark.parametrize("mode,storage", [("fast", "fp32"), ("exact", "fp32"), ("fast", "fp16")])
@pytest.mark.parametrize("kind", KINDS)
def test_inline_equals_separate(kind, mode, storage):
    pb = build(kind)
    want, wf = run(pb, mode, storage, 4)
    assert np.abs(want).max() > 0
    for rows, zchunk in ((2, 4), (4, 7), (1, 64)):
        got, gf = run(pb, mode, storage, 1, rows, zchunk)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (kind, rows, zchunk)
        for a, b in zip(gf, wf):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["fp32", "fp16"])
def test_batch_inline_equals_alone(storage):
    """Every kind of source in one batch, inline and separate side by side,
    with a grid that joins late."""
    from semba_fdtd_amd.batch import Batch
    pbs = [build(k, nx=60 + 3 * q) for q, k in enumerate(KINDS)]
    alone = [run(pb, "fast", storage, 4)[0] for pb in pbs]
    b = Batch()
    sol = [sf.Solver(pb, storage=storage) for pb in pbs]
    for s in sol[:-1]:
        b.admit(s)
    b.step(5)
    b.admit(sol[-1])
    b.step(STEPS - 5)
    for slot, s in list(b.members.items()):
        if s is sol[-1]:
            b.retire(slot)
    sol[-1].run(5)
    for s, want, kind in zip(sol, alone, KINDS):
        got = s.probes()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), kind
    b.close()
