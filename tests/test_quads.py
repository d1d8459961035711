"""The four-cell face passes against the general path (one entry point per
reference routine, one cell per lane, sources in launches of their own): the
same bits at the widths where a row's vectors, a wave's lanes, a tile's rows or
a slab end, on every box layout of the plan."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P

STEPS = 24
SPLIT = ("advance_e_yee", "advance_e_cpml", "advance_e_dispersive", "advance_planewave_e",
         "advance_nodal_e", "advance_h_yee", "advance_h_cpml", "advance_h_dispersive",
         "advance_planewave_h", "advance_nodal_h", "advance_mur")


def build(n, L, wave=False, disp=False, mur=None):
    pb = P.scatterer_problem(n=n, L=L, nsteps=STEPS, disp=disp, mdisp=disp, mur=mur)
    if wave:
        q = np.arange(STEPS + 5)
        ev = (np.sin(q / 3.0) * (1 - np.exp(-q / 2.0))).astype(np.float32)
        lo, hi = [L[a][0] + 1 for a in range(3)], [n[a] - L[a][1] - 2 for a in range(3)]
        box = tuple(v for a in range(3) for v in (lo[a], hi[a]))
        pb.planewaves = [P.PlaneWave(box, [(0.48, 0.64, 0.6)], [(0.8, -0.6, 0.0)], ev,
                                     float(np.float32(pb.dt)))]
    return pb


def start(s, pb):
    for c in range(6):
        ex = P.alloc_extent(c, (pb.nx, pb.ny, pb.nz))
        a = np.zeros(ex[::-1], np.float32)
        a[1:-1, 1:-1, 1:-1] = np.random.default_rng(c).standard_normal(
            [v - 2 for v in ex[::-1]]) * (1.0 if c < 3 else 1 / 377.0)
        s.set_field(c, a)


def split(pb, mode):
    s = sf.Solver(pb, mode=mode)
    start(s, pb)
    for n in range(STEPS):
        for name in SPLIT:
            f = getattr(s.lib, "fdtd_" + name)
            rc = f(s.h, n) if "planewave" in name or "nodal" in name else f(s.h)
            assert rc == 0, name
    return [s.field(c) for c in range(6)]


def fused(pb, mode, storage="fp32", tiling=None):
    s = sf.Solver(pb, mode=mode, storage=storage)
    if tiling:
        s.set_tiling(*tiling)
    start(s, pb)
    s.run(STEPS)
    return [s.field(c) for c in range(6)]


def same(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))


NONE = ((0, 0),) * 3
CASES = [((nx, 13, 11), NONE, False, False) for nx in (9, 10, 11, 12, 63, 64, 255, 256, 257)] + [
    ((nx, 15, 14), ((lx, hx), (3, 2), (2, 3)), True, False)
    for nx, lx, hx in ((15, 4, 4), (16, 5, 3), (17, 3, 6), (18, 1, 0), (19, 0, 7), (67, 8, 8), (258, 10, 9))] + [
    ((20, 15, 14), ((4, 4), (0, 0), (0, 0)), True, False),       # x slabs alone
    ((20, 18, 14), ((0, 0), (4, 5), (0, 0)), True, False),
    ((20, 15, 18), ((0, 0), (0, 0), (5, 4)), True, False),
    ((33, 26, 24), ((4, 5), (3, 4), (5, 3)), False, True),       # pole media
    ((33, 26, 24), ((4, 5), (3, 4), (5, 3)), True, True),
    ((130, 40, 31), ((8, 8), (8, 8), (8, 8)), True, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["fast", "exact"])
@pytest.mark.parametrize("n,L,wave,disp", CASES)
def test_quads_equal_split(n, L, wave, disp, mode):
    print(n, L, wave, disp, mode, flush=True)
    pb = build(n, L, wave, disp)
    want = split(pb, mode)
    assert np.abs(want[0]).max() > 0
    assert same(fused(pb, mode), want)
    for tiling in ((1, 5, 4), (4, 64, 4)):
        assert same(fused(pb, mode, tiling=tiling), want), tiling


@pytest.mark.gpu
@pytest.mark.parametrize("n,L,wave,disp", CASES[3:])
def test_quads_equal_one_cell_binary16(n, L, wave, disp):
    print(n, L, wave, disp, flush=True)
    pb = build(n, L, wave, disp)
    want = fused(pb, "fast", "fp16", (2, 4, 1))
    assert same(fused(pb, "fast", "fp16"), want)
    assert same(fused(pb, "fast", "fp16", (4, 3, 4)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("n,L", [((9, 20, 19), ((3, 3), (0, 0), (0, 0))),    # a vector would meet both slabs
                                 ((20, 9, 19), ((4, 4), (4, 4), (4, 4))),    # no row clear of the y slabs
                                 ((5,) * 3, NONE), ((7,) * 3, NONE)])
def test_grids_without_interior(n, L):
    print(n, L, flush=True)
    if n[0] < 8:
        pb = P.cavity_problem(n=n[0], nsteps=STEPS)
    else:
        pb = build(n, NONE)
        pb.cpml_layers = [list(v) for v in L]
    want = split(pb, "fast")
    assert same(fused(pb, "fast"), want)
    assert same(fused(pb, "fast", tiling=(2, 4, 4)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["fp32", "fp16"])
@pytest.mark.parametrize("narrow", [False, True])
def test_batch_quads_equal_alone(storage, narrow):
    """Grids of every layout in one batch; with a grid the four-cell passes
    cannot run (narrow) the whole batch runs one cell per lane."""
    from semba_fdtd_amd.batch import Batch
    pbs = [build(*CASES[q]) for q in (2, 9, 12, 15, 16, 17, 18, 20, 21)]
    if narrow:
        pbs.append(build((9, 20, 19), NONE))
        pbs[-1].cpml_layers = [[3, 3], [0, 0], [0, 0]]
    want = [fused(pb, "fast", storage, (2, 4, 1)) for pb in pbs]
    for tiling in ((4, 16, 0, 1), (2, 5, 0, 4)):
        b = Batch()
        b.set_tiling(*tiling)
        sol = [sf.Solver(pb, storage=storage) for pb in pbs]
        for s, pb in zip(sol, pbs):
            start(s, pb)
            b.admit(s)
        b.step(STEPS)
        for q, s in enumerate(sol):
            assert same([s.field(c) for c in range(6)], want[q]), (tiling, q)
        b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("wave", [False, True])
def test_observation_in_the_passes(wave):
    """Probes of all components and frequency-domain boxes of H before E, in
    runs of the 16-step and the one-step graph, against call by call."""
    pb = build((67, 15, 14), ((8, 8), (3, 2), (2, 3)), wave)
    pb.dfts = [P.DftBox(1, (0, 66, 3, 6, 4, 6), (3, 1, 1), [0.7e9, 1.9e9]),
               P.DftBox(0, (1, 60, 2, 9, 3, 3), (2, 2, 1), [1.1e9])]
    a, b = sf.Solver(pb), sf.Solver(pb)
    for n in (1, 5, 6):
        a.run(n)
    for _ in range(12):
        b.step()
    assert np.array_equal(a.probes().view(np.uint32), b.probes().view(np.uint32))
    for x, y in zip(a.dft_sums(), b.dft_sums()):
        assert np.abs(x).max() > 0 and np.array_equal(x.view(np.uint64), y.view(np.uint64))
    a.set_graph_steps(4)
    a.run(9)
    for _ in range(9):
        b.step()
    assert np.array_equal(a.probes().view(np.uint32), b.probes().view(np.uint32))
