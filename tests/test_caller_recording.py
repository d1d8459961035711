"""Steps that a caller records on the grid's stream (hipStreamBeginCapture
around the step calls) and replays, mixed with direct calls and runs: the same
bits as the same steps called directly.  A recorded call has to do by itself
what it does when called, whatever ran or was replayed in between."""
import ctypes as C

import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd._lib import i32p, ptr

pytestmark = pytest.mark.gpu

STEPS = 30
PRIO = np.array([1000, 0, 20], np.int32)


class Recorder:
    """A stream of the library's own HIP runtime, and recordings of it."""

    def __init__(self):
        self.hip = sf.load_library()     # its dependencies resolve through it
        self.stream = C.c_void_p()
        self._do("hipStreamCreateWithFlags", C.byref(self.stream), 1)
        self.graphs = []

    def _do(self, name, *args):
        f = getattr(self.hip, name)
        f.restype = C.c_int
        rc = f(*args)
        assert rc == 0, (name, rc)

    def record(self, calls):
        graph, ex = C.c_void_p(), C.c_void_p()
        self._do("hipStreamBeginCapture", self.stream, 1)
        try:
            calls()
        finally:
            self._do("hipStreamEndCapture", self.stream, C.byref(graph))
        self._do("hipGraphInstantiate", C.byref(ex), graph, None, None, C.c_size_t(0))
        self.graphs.append((graph, ex))
        return ex

    def replay(self, ex):
        self._do("hipGraphLaunch", ex, self.stream)

    def close(self):
        self._do("hipStreamSynchronize", self.stream)
        for graph, ex in self.graphs:
            self._do("hipGraphExecDestroy", ex)
            self._do("hipGraphDestroy", graph)
        self._do("hipStreamDestroy", self.stream)


@pytest.fixture
def rec():
    r = Recorder()
    yield r
    r.close()


def step(s, n):
    for name in ("advance_e", "advance_h", "update_observation"):
        assert getattr(s.lib, "fdtd_" + name)(s.h, n) == 0, s.lib.fdtd_last_error(s.h)


def fields(s):
    return [s.field(c) for c in range(6)]


def same(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))


def wave_problem(nodal=False):
    pb = P.scatterer_problem(n=(40, 30, 28), L=((4, 5), (3, 4), (5, 3)), nsteps=4 * STEPS, disp=False)
    if not nodal:
        pb.nodal = []
    q = np.arange(STEPS + 5)
    ev = (np.sin(q / 3.0) * (1 - np.exp(-q / 2.0))).astype(np.float32)
    pb.planewaves = [P.PlaneWave((6, 33, 5, 24, 7, 23), [(0.48, 0.64, 0.6)], [(0.8, -0.6, 0.0)], ev,
                                 float(np.float32(pb.dt)))]
    pb.probes = []
    return pb


@pytest.mark.parametrize("tiling", [None, (2, 4, 1)])
@pytest.mark.parametrize("then", ["advance", "run"])
def test_direct_steps_after_a_replay(rec, tiling, then):
    """Ten steps called directly leave the plane wave's next terms behind; a
    replay of recorded steps writes the terms of its own.  The steps that
    follow need theirs."""
    pb = wave_problem()

    def grid(**kw):
        s = sf.Solver(pb, **kw)
        if tiling:
            s.set_tiling(*tiling)
        return s

    ref = grid()
    for n in range(16):
        step(ref, n)
    want = fields(ref)
    s = grid(stream=rec.stream)
    start = s.save_state()
    for n in range(10):
        step(s, n)
    s.load_state(start)
    ten = rec.record(lambda: [step(s, n) for n in range(10)])
    for _ in range(3):
        s.load_state(start)
        for n in range(10):
            step(s, n)
        s.load_state(start)
        rec.replay(ten)
        if then == "run":
            assert s.lib.fdtd_run(s.h, 10, 6) == 0
        else:
            for n in range(10, 16):
                step(s, n)
        assert np.abs(want[0]).max() > 0
        assert same(fields(s), want)
    s.close()


def test_half_steps_after_a_replay(rec):
    """A recorded step replayed between the halves of a direct one (on a
    saved state of its own) leaves the second half its terms."""
    pb = wave_problem()
    ref = sf.Solver(pb)
    for n in range(12):
        step(ref, n)
    want = fields(ref)
    s = sf.Solver(pb, stream=rec.stream)
    for n in range(10):
        step(s, n)
    three = rec.record(lambda: step(s, 3))
    assert s.lib.fdtd_advance_e(s.h, 10) == 0
    mid = s.save_state()
    rec.replay(three)
    s.load_state(mid)
    assert s.lib.fdtd_advance_h(s.h, 10) == 0
    step(s, 11)
    assert same(fields(s), want)
    s.close()


@pytest.mark.parametrize("tiling", [None, (2, 4, 1)])
def test_recording_after_a_media_change(rec, tiling):
    """Media written since the last step, the sources as they were: the step
    calls can be recorded at once."""
    pb = wave_problem()
    s = sf.Solver(pb, stream=rec.stream)
    ref = sf.Solver(pb)
    if tiling:
        s.set_tiling(*tiling)
    for q in (s, ref):
        for n in range(12):
            step(q, n)
        assert q.lib.fdtd_media_paint_box(q.h, 12, 20, 10, 16, 9, 15, 2, 3, ptr(PRIO, i32p)) == 0
    two = rec.record(lambda: [step(s, n) for n in (12, 13)])
    rec.replay(two)
    for n in (12, 13):
        step(ref, n)
    got, want = fields(s), fields(ref)
    assert np.abs(want[0]).max() > 0 and same(got, want), tiling
    s.close()


@pytest.mark.parametrize("tiling", [None, (2, 4, 1)])
def test_recording_outlives_what_drops_the_graphs(rec, tiling):
    """Calls that only drop the library's own recorded steps (here the step
    mode set again) leave a caller's recording what it reads: the sources'
    tables stay where they are."""
    pb = wave_problem(nodal=True)

    def grid(**kw):
        s = sf.Solver(pb, **kw)
        if tiling:
            s.set_tiling(*tiling)
        return s

    ref = grid()
    for n in range(16):
        step(ref, n)
    want = fields(ref)
    s = grid(stream=rec.stream)
    start = s.save_state()
    for n in range(10):
        step(s, n)
    s.load_state(start)
    ten = rec.record(lambda: [step(s, n) for n in range(10)])
    s.set_step_mode(0, 16)
    step(s, 0)
    others = [sf.Solver(P.scatterer_problem(nsteps=20)) for _ in range(3)]
    for q in others:
        q.run(5)
    for _ in range(2):
        s.load_state(start)
        rec.replay(ten)
        for n in range(10, 16):
            step(s, n)
        assert same(fields(s), want)
    s.close()


@pytest.mark.parametrize("tiling", [None, (2, 4, 1)])
def test_direct_steps_after_a_recording_not_replayed(rec, tiling):
    """What a recording would renew has not been renewed until it is replayed:
    media written, steps recorded, and direct steps instead."""
    pb = wave_problem()
    s, ref = sf.Solver(pb, stream=rec.stream), sf.Solver(pb)
    if tiling:
        s.set_tiling(*tiling)
    for q in (s, ref):
        for n in range(12):
            step(q, n)
        assert q.lib.fdtd_media_paint_box(q.h, 8, 30, 6, 22, 8, 20, 2, 3, ptr(PRIO, i32p)) == 0
    two = rec.record(lambda: [step(s, n) for n in (12, 13)])
    for n in range(12, 16):
        step(s, n)
    for n in range(12, 16):
        step(ref, n)
    want = fields(ref)
    assert np.abs(want[0]).max() > 0 and same(fields(s), want)
    start = s.save_state()
    for k in range(2):                               # and the recording itself
        s.load_state(start)
        rec.replay(two)
        if k == 0:
            again = fields(s)
    assert same(fields(s), again)
    s.close()


def test_granular_calls_recorded_first(rec):
    """The granular calls first made inside a recording, on a grid whose steps
    so far were fused ones; recorded after a media change; and directly."""
    pb = wave_problem(nodal=True)
    names = ("advance_e_yee", "advance_e_cpml", "advance_planewave_e", "advance_nodal_e",
             "advance_h_yee", "advance_h_cpml", "advance_planewave_h", "advance_nodal_h")

    def granular(s, n):
        for name in names:
            f = getattr(s.lib, "fdtd_" + name)
            assert (f(s.h, n) if "planewave" in name or "nodal" in name else f(s.h)) == 0, name

    s, ref = sf.Solver(pb, stream=rec.stream), sf.Solver(pb)
    for q in (s, ref):
        for n in range(12):
            step(q, n)
    two = rec.record(lambda: [granular(s, n) for n in (12, 13)])
    rec.replay(two)
    for n in range(14, 17):
        granular(s, n)
    pb2 = rec.record(lambda: granular(s, 17))
    rec.replay(pb2)
    for n in range(12, 18):
        step(ref, n)
    want = fields(ref)
    assert np.abs(want[0]).max() > 0 and same(fields(s), want)
    s.close()
