"""Sources inside the face passes against the launches of their own that the
granular calls run (k_tfsf_list, k_nodal): the same passes with the inline
sources off are the reference.  Four cells per lane and one, both arithmetic
modes and binary16 storage, whose separate launches round each source's store
once; waves along every axis, whose terms are held one per line."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from test_inline_sources import KINDS, STEPS, build, wave

pytestmark = pytest.mark.gpu

AXES = {"+x": ((1.0, 0.0, 0.0), (0.0, 0.6, 0.8)), "-y": ((0.0, -1.0, 0.0), (0.8, 0.0, 0.6)),
        "+z": ((0.0, 0.0, 1.0), (0.6, -0.8, 0.0)), "xy": ((0.6, 0.8, 0.0), (0.0, 0.0, 1.0)),
        "yz": ((0.0, 0.6, -0.8), (1.0, 0.0, 0.0)), "xyz": ((0.48, 0.64, 0.6), (0.8, -0.6, 0.0))}
# the kinds whose sources the passes take in both halves (poles keep others out)
INLINE = {"plain", "nodal_shared", "modes"} | set(AXES)


def problem(kind, nx=70):
    if kind in KINDS:
        return build(kind, nx)
    pb = build("plain", nx)
    if kind in AXES:
        p, e = AXES[kind]
        pb.planewaves = [wave(pb, (6, nx - 7, 5, 20, 7, 19), p, e)]
    else:                            # two modes: along z, and across
        w = wave(pb, (6, nx - 7, 5, 20, 7, 19))
        pb.planewaves = [P.PlaneWave(w.box, [AXES[k][0] for k in ("+z", "xy")],
                                     [AXES[k][1] for k in ("+z", "xy")], w.evol, w.deltaevol)]
    return pb


def run(pb, mode, storage, inline, tiling=None):
    s = sf.Solver(pb, mode=mode, storage=storage)
    assert s.lib.sfd_set_inline_sources(s.h, int(inline)) == 0
    if tiling:
        s.set_tiling(*tiling)
    on = s.lib.sfd_inline_sources(s.h)
    assert on >= 0 and (inline or on == 0)
    s.run(STEPS - 1)
    s.step()
    r = [s.probes()] + [s.field(c) for c in range(6)]
    s.close()
    return on, r


def same(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))


@pytest.mark.parametrize("mode,storage", [("fast", "fp32"), ("exact", "fp32"), ("fast", "fp16")])
@pytest.mark.parametrize("kind", KINDS + list(AXES) + ["modes"])
def test_inline_equals_launches_of_their_own(kind, mode, storage):
    print(kind, mode, storage, flush=True)
    pb = problem(kind)
    _, want = run(pb, mode, storage, False)
    assert np.abs(want[0]).max() > 0 and np.isfinite(want[0]).all()
    assert same(run(pb, mode, storage, False, (2, 4, 1))[1], want)
    for tiling in (None, (2, 5, 4), (2, 4, 1)):
        on, got = run(pb, mode, storage, True, tiling)
        assert on == 3 or kind not in INLINE
        assert same(got, want), tiling


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
@pytest.mark.parametrize("xcells", [1, 4])
def test_batch_inline_equals_launches_of_their_own(storage, xcells):
    from semba_fdtd_amd.batch import Batch
    kinds = KINDS + list(AXES)
    pbs = [problem(k, nx=60 + 3 * q) for q, k in enumerate(kinds)]
    b = Batch(rows=2, zchunk=5, xcells=xcells)
    sol = [sf.Solver(pb, storage=storage) for pb in pbs]
    for s in sol:
        b.admit(s)
    b.step(STEPS)
    for s, pb, kind in zip(sol, pbs, kinds):
        want = run(pb, "fast", storage, False)[1]
        assert same([s.probes()] + [s.field(c) for c in range(6)], want), kind
    b.close()
