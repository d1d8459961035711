"""One-launch steps with plain tiles merged over several z chunks (what large
grids run) and unmerged (mid-size ones), class kernels one after another and
in branches of the recorded step, on grids deeper than a chunk: the bits of
the two passes, whatever the rule would choose."""
import numpy as np
import pytest

import oracle
import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from test_step_kernel import VEC_CASES

pytestmark = pytest.mark.gpu

SHAPES = [(m, f) for m in (1, 0) for f in (0, 1)]


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def tiles(s):
    n = np.zeros(17, np.int32)
    assert s.lib.sfd_step_tiles(s.h, n.ctypes) == 0
    return n


def stepped(pb, ns, mode, rows, kc, merge, fork, init=()):
    s = sf.Solver(pb, mode=mode)
    for c, a in enumerate(init):
        s.set_field(c, a)
    s.set_step_mode(rows, kc)
    assert s.lib.sfd_set_step_plan(s.h, merge, fork) == 0
    s.run(ns)
    return s


@pytest.mark.parametrize("name", list(VEC_CASES))
def test_every_shape_equals_oracle(name):
    pb = VEC_CASES[name]()
    ns = pb.nsteps_max
    ref = oracle.Oracle(pb)
    want = ref.run(ns)
    plain = {}
    for rows, kc in ((16, 4), (8, 7)):
        for merge, fork in SHAPES:
            print(name, rows, kc, merge, fork, flush=True)
            s = stepped(pb, ns, "exact", rows, kc, merge, fork)
            n = tiles(s)
            plain[merge] = n[0] + n[8]
            assert np.array_equal(bits(s.probes()), bits(want))
            for c in range(6):
                assert np.array_equal(bits(s.field(c)), bits(ref.fields[c])), (rows, kc, merge, fork, c)
            s.close()
        assert plain[1] < plain[0] or pb.nz + 1 <= kc, (plain, kc)   # tiles did merge


@pytest.mark.parametrize("mode", ["exact", "fast"])
def test_open_scatterer_equals_two_passes(mode):
    """256^3 with CPML, plane wave and sphere, every field set: merged tiles of
    64 planes."""
    ns = 24
    pb = P.open_scatterer_problem(n=256, nsteps=ns, spread=4, delay=8)
    a = sf.Solver(pb, mode=mode)
    init = []
    for c in range(6):
        f = np.zeros(pb.alloc_shape, np.float32)
        f[1:-2, 1:-2, 1:-2] = np.random.default_rng(c).standard_normal(
            [v - 3 for v in pb.alloc_shape], np.float32) * np.float32(1.0 if c < 3 else 1 / 377.0)
        init.append(f)
        a.set_field(c, f)
    a.run(ns)
    want = [a.field(c) for c in range(6)]
    assert all(np.abs(w).max() > 0 and np.isfinite(w).all() for w in want)
    for merge, fork in SHAPES:
        print(mode, merge, fork, flush=True)
        s = stepped(pb, ns, mode, 16, 16, merge, fork, init)
        assert np.array_equal(bits(s.probes()), bits(a.probes()))
        for c in range(6):
            assert np.array_equal(bits(s.field(c)), bits(want[c])), (merge, fork, c)
        s.close()
    a.close()
