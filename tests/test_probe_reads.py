"""fdtd_read_probes at sizes around the samples it reads along with the count:
every sample arrives, and a large read needs no memory of its own size."""
import ctypes as C

import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd._lib import f32p, ptr

pytestmark = pytest.mark.gpu


def grid(nprobe, steps):
    pb = P.cavity_problem(n=12, nsteps=steps)
    rng = np.random.default_rng(nprobe)
    pb.probes = [(int(rng.integers(0, 6)),) + tuple(int(v) for v in rng.integers(1, 11, 3))
                 for _ in range(nprobe)]
    return sf.Solver(pb, probe_buffer=steps)


def read(s, room, out=None):
    out = np.full((room, s.nprobe), np.nan, np.float32) if out is None else out
    k = C.c_int32()
    rc = s.lib.fdtd_read_probes(s.h, ptr(out, f32p), room, C.byref(k))
    return rc, k.value, out


@pytest.mark.parametrize("nprobe", [1, 15, 16, 4095, 4096, 4097])
def test_reads_of_any_length(nprobe):
    """4096 values ride with the count: reads ending before, at and after
    them, an empty one, and one without the room."""
    per = max(4096 // nprobe, 1)
    total = 3 * per + 4
    s, ref = grid(nprobe, total), grid(nprobe, total)
    ref.run(total)
    want = ref.probes()
    n = 0
    for steps in (per, per - 1, 0, per + 1):
        if steps:
            assert s.lib.fdtd_run(s.h, n, steps) == 0
        if steps > 1:
            assert read(s, steps - 1)[:2] == (-1, 0)
        rc, k, got = read(s, steps + 1)
        assert rc == 0 and k == steps
        assert np.array_equal(got[:k].view(np.uint32), want[n:n + k].view(np.uint32))
        assert np.isnan(got[k:]).all()
        n += steps
    assert read(s, 1)[:2] == (0, 0)


def peak():
    with open("/proc/self/status") as f:
        return next(int(v.split()[1]) for v in f if v.startswith("VmHWM")) << 10


def test_large_read_in_place():
    nprobe, steps = 8000, 2000                       # 64 MB
    s = grid(nprobe, steps)
    out = np.ones((steps, nprobe), np.float32)
    for k in (16, 400):                              # (the runtime's own staging)
        assert s.lib.fdtd_run(s.h, 0, k) == 0 and read(s, steps, out)[:2] == (0, k)
    assert s.lib.fdtd_run(s.h, 0, steps) == 0
    s.synchronize()
    before = peak()
    assert read(s, steps, out)[:2] == (0, steps)
    assert peak() - before < out.nbytes // 2
