"""The four-cell passes over grids with large media tables (four rows of a
block share one): the bits of the one-cell passes, alone and in a batch with
grids of few media, up to the largest table the passes stage."""
import numpy as np
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd.batch import Batch
from test_quads import fused, same, start

pytestmark = pytest.mark.gpu


def problem(nm, n=(37, 15, 12)):
    """Random media everywhere inside."""
    base = P.scatterer_problem(n=n, L=((4, 5), (3, 2), (2, 3)), nsteps=24, disp=False)
    rng = np.random.default_rng(nm)
    mi = base.mi.copy()
    inner = tuple(slice(3, v - 2) for v in mi.shape[1:])
    for c in range(6):
        mi[c][inner] = rng.integers(1, nm + 1, size=mi[c][inner].shape).astype(mi.dtype)
    return P.Problem(*n, epr=[1.0, 1.0] + list(rng.uniform(1.0, 6.0, nm - 1)),
                     sigma=[0.0, 0.0] + list(rng.uniform(0.0, 0.2, nm - 1)), mur=[1.0] * (nm + 1),
                     sigmam=[0.0] * (nm + 1), kind=[P.KIND_PEC] + [0] * nm, mi=mi, D=base.D, dt=base.dt,
                     cpml_layers=base.cpml_layers, cpml_order=base.cpml_order,
                     cpml_refl=base.cpml_refl, nodal=base.nodal, probes=base.probes,
                     nsteps_max=24, name=f"media{nm}")


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
@pytest.mark.parametrize("nm,rows", [(255, 1), (256, 4), (1000, 4), (4095, 4)])
def test_large_tables_share_rows(nm, rows, storage):
    pb = problem(nm)
    assert sf.Solver(pb, storage=storage).get_tiling() == (rows, 1, 4)
    want = fused(pb, "fast", storage, (2, 4, 1))
    assert np.isfinite(want[0]).all() and np.abs(want[0]).max() > 0
    assert same(fused(pb, "fast", storage), want)


@pytest.mark.parametrize("storage", ["fp32", "fp16"])
def test_batch_with_a_large_table(storage):
    pbs = [problem(3, (20, 15, 14)), problem(2000), problem(12, (64, 13, 15))]
    want = [fused(pb, "fast", storage, (2, 4, 1)) for pb in pbs]
    b = Batch()
    sol = [sf.Solver(pb, storage=storage) for pb in pbs]
    for s, pb in zip(sol, pbs):
        start(s, pb)
        b.admit(s)
    b.step(24)
    for s, w in zip(sol, want):
        assert same([s.field(c) for c in range(6)], w)
    b.close()
