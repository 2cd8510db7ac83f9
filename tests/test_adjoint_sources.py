"""The cell sources' reverse pass (source_back, eddy_back of
adjoint_point.hpp, compiled for the host) against one-lane dual passes over
all of the sources' inputs: every mass-transfer model, SST with each length
scale, the BDF term, the eddy viscosity as a state function.  Both follow the
same selections and differ by rounding only: 1e-10 of the largest change any
input's own size makes."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
TOL = 1e-10


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("adjsrc") / "libsrccheck.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-ffp-contract=off", "-std=c++17",
                    "-fPIC", "-shared", "-w", os.path.join(HERE, "native", "srccheck.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.mark.parametrize("models,ncav,iturb,ides,nsteady,eddy", [
    (0, 0, -3, 0, 0, 0), (0, 1, -2, 0, 0, 0), (0, 0, 0, 0, 0, 0), (0, 1, 0, 0, 2, 0), (0, 1, 0, 0, 1, 1), (0, 0, -2, 0, 1, 0),
    (1, 2, -2, 0, 0, 0), (1, 3, 0, 0, 2, 1), (1, 4, -2, 0, 0, 0), (1, 5, 0, 0, 0, 0),
    (1, 0, 0, 1, 0, 0), (1, 1, 0, 2, 0, 1), (1, 0, 0, 3, 2, 0), (1, 1, 0, 4, 0, 0)])
def test_cell_sources(L, models, ncav, iturb, ides, nsteady, eddy):
    rng = np.random.default_rng(1000 * ncav + 100 * ides + 10 * nsteady + eddy - iturb)
    for trial in range(300):
        z = np.zeros(31)
        z[0] = rng.uniform(-4.5e3, 4e4)                      # around the vapour pressure with p_ref = 5e3
        z[1:4] = rng.standard_normal(3) * 10
        z[4] = rng.uniform(290, 320)
        z[5:7] = rng.uniform(1e-6, 0.1, 2)
        z[7], z[8] = 10.0 ** rng.uniform(-4, 0), 10.0 ** rng.uniform(1, 5)
        z[9:24] = rng.standard_normal(15) * 10.0 ** rng.uniform(0, 4)
        z[24], z[25], z[26], z[27] = rng.uniform(1, 1000), rng.uniform(1e5, 3e5), rng.uniform(5e-4, 1.5e-3), 10.0 ** rng.uniform(-4, -1)
        z[28:31] = 10.0, 2e-5, 100.0
        d = np.zeros(13)
        d[:] = rng.uniform(0.5, 2.0, 13)
        f = rng.standard_normal(18) * 1e-4
        rb = rng.standard_normal(9) / np.array([1, 10, 10, 10, 1e5, 1, 1, 1, 1])
        d[0], d[1], d[11] = z[24], z[25], z[26]              # rho, h, mu
        rev, dual = np.zeros(31), np.zeros(31)
        L.sc_source(models, ncav, iturb, ides, nsteady, dp(z), dp(d), dp(f), C.c_double(1e-7), C.c_double(10.0 ** rng.uniform(-6, -2)),
                    dp(rb), C.c_double(rng.standard_normal() if eddy else 0.0), dp(rev), dp(dual))
        ref = np.maximum(np.abs(z), 1e-3)
        if ncav > 3 or ncav == 0:                            # the scales of the other models are not asked for
            assert not np.any(rev[28:])
            dual[28:] = 0.0
        r, u = rev * ref, dual * ref
        assert np.all(np.isfinite(r)) and np.max(np.abs(r - u)) <= TOL * np.max(np.abs(u)), (trial, z, rev, dual)
