"""The sweeps' cell records and their stage at the edges of the 4 x 4 pencil
tiles (tiles cut off in j, in k and in both, pencils shorter than the stage's
ring, absent neighbours on every side, blocks of different sizes) against the
oracle, to the parity bar of 1e-11."""
import numpy as np
import pytest

from parity import interior, pair, rel_err

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (4, 4, 4), (5, 5, 3), (6, 4, 7), (9, 9, 4), (21, 6, 5)]


@pytest.mark.parametrize("turbulent", [False, True])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("cut", [False, True])
def test_step_at_tile_edges(pkg, orc, size, turbulent, cut):
    print(f"size {size} turbulent {turbulent} cut {cut}", flush=True)
    if cut and size[0] < 6:
        pytest.skip("a block has at least three cells in i")
    case = pkg.cases.config2(*size) if turbulent else pkg.cases.config1(*size)
    case.params["cav_clip"] = 1
    if cut:
        case = pkg.cases.split_i(case, [4])
    s, o = pair(pkg, orc, case)
    for it in (1, 2):
        s.timeinteg(1, it, 0.0)
        o.timeinteg(1, it, 0.0)
    for ib in range(len(case.blocks)):
        a = interior(case, ib, s.get_state(ib)[0], case.npv)
        b = interior(case, ib, o.get_state(ib)[0], case.npv)
        assert np.all(rel_err(a, b) < 1e-11), rel_err(a, b)
    s.close()
