"""fdtd_device_bytes counts what a grid holds: tables built again after a
change take the place of the old ones, and a batch's tables are the batch's."""
import pytest

import semba_fdtd_amd as sf
from semba_fdtd_amd import problem as P
from semba_fdtd_amd.batch import Batch

pytestmark = pytest.mark.gpu


def grid():
    pb = P.scatterer_problem(nsteps=60)          # poles, nodal E and H sources
    pb.nodal[0].box = (8, 9, 9, 10, 14, 14)      # clear of the pole-state boxes: inline
    return sf.Solver(pb)


@pytest.mark.parametrize("what", ["tiling", "media", "step", "batch"])
def test_bytes_stay_as_tables_are_rebuilt(what):
    s = grid()
    b = Batch()

    def cycle():
        if what == "tiling":
            for t in ((2, 4, 4), (2, 4, 1)):
                s.set_tiling(*t)
                s.run(2)
        elif what == "media":
            assert s.lib.fdtd_set_media_index(s.h, 0, media) == 0
            s.run(2)
        elif what == "step":
            for rows in (8, 0):
                s.set_step_mode(rows, 8)
                s.run(2)
        else:
            slot = b.admit(s)
            b.step(2)
            b.retire(slot)

    from semba_fdtd_amd._lib import i16p, ptr
    m = P.to_alloc_box(s.pb.mi[0], 0, s.n3)
    media = ptr(m, i16p)
    cycle()
    held = s.device_bytes
    for _ in range(3):
        cycle()
    assert s.device_bytes == held
    b.close()
    s.close()
