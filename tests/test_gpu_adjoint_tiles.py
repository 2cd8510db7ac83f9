"""The adjoint's stencil pass at the edges of its tiles, against central
differences of the residual over every ghosted cell (as
test_gpu_adjoint.py, with its tolerance).  The third-order limiter without
bounds (9) keeps the reconstruction smooth, so directions settle on grids of
any size: grids below, at and above one tile of either shape in each direction,
and one with enough of the larger tiles to take them."""
import zlib

import numpy as np
import pytest

import test_gpu_adjoint as tga
from test_gpu_adjoint import _close_contexts  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("muscl", [1, 2])
@pytest.mark.parametrize("size", [(11, 6, 4), (12, 11, 4), (28, 12, 11), (29, 13, 20), (118, 50, 49)],
                         ids=lambda s: "x".join(map(str, s)))
def test_stencil_pass_matches_central_differences(pkg, size, muscl):
    print(f"case {size} muscl {muscl}", flush=True)
    name = f"tiles{size}{muscl}"
    case, s, pvs, fr = tga.prepared(pkg, name, make=lambda: pkg.cases.bump_case(*size, False, False, 1, muscl, 9, cfl=1.0, seed=9))
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    rb = tga.seeds(case, s.residual_of(pvs, fr["mut"], fr["qq"]), rng)
    pb, _ = s.rhs_vjp(rb)
    tga.check_directions(lambda p: s.residual_of(p, fr["mut"], fr["qq"]), pvs, pb, rb, tga.directions(case, pvs, rng, 4), 3)
    s.close()
