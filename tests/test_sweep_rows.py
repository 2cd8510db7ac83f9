"""The sweeps' row form (sweep_rows.hpp, compiled for the host with sixteen
emulated lanes) against the row-by-row Jacobian products and D^-1 that the
other host tests hold against the oracle: the same bits, for both sweeps, both
systems, and neighbours within the tile and across its edge."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import physhost as H

HERE = os.path.dirname(os.path.abspath(__file__))


def dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rows") / "librowcheck.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-ffp-contract=off", "-std=c++17",
                    "-fPIC", "-shared", "-w", os.path.join(HERE, "native", "rowcheck.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def problem(pkg, npv):
    case = (pkg.cases.config1 if npv == 7 else pkg.cases.config2)(8, 6, 6)
    iv, dv = H.par_arrays(case.cfg_dict())
    return case, iv, dv


def cells(pkg, rng, npv, pref):
    """Four cells: state, properties, eddy viscosity, volume, faces."""
    out = np.zeros((4, 42))
    for c in out:
        c[:9] = [rng.uniform(-3e4, 3e4), rng.uniform(-15, 15), rng.uniform(-3, 3), rng.uniform(-3, 3), rng.uniform(290, 310),
                 0.0 if npv == 7 else rng.choice([0.0, rng.uniform(0, 1e-3), rng.uniform(0, 0.5)]), 0.0,
                 rng.uniform(1e-4, 0.1) if npv == 9 else 0.0, rng.uniform(10, 1e4) if npv == 9 else 0.0]
        dvv, tv = pkg.eos_host(c[0] + pref, c[4], c[5], c[6])
        c[9:22] = H.compact(dvv[0], tv[0])
        c[22] = rng.uniform(1e-5, 1e-2) if npv == 9 else 0.0
        c[23] = rng.uniform(1e-9, 1e-6)
        c[24:] = rng.standard_normal(18) * 1e-4
    return out


def step(L, iv, dv, fwd, edge, c, rng):
    cc, tt, res = rng.standard_normal(4) * 1e5, rng.standard_normal(4) * 1e2, rng.standard_normal(9)
    x, o = rng.standard_normal((3, 9)), np.zeros((6, 9))
    c = np.ascontiguousarray(c)
    L.rc_step(iv.ctypes.data_as(C.POINTER(C.c_int)), dp(dv), fwd, edge, dp(c), C.c_double(rng.uniform(1e-5, 1e-2)), dp(cc), dp(tt),
              dp(res), dp(x), *(dp(r) for r in o))
    return o


@pytest.mark.parametrize("npv", [7, 9])
@pytest.mark.parametrize("fwd", [1, 0])
@pytest.mark.parametrize("edge", [0, 1])
def test_rows_of_lanes_bit_exact(L, pkg, npv, fwd, edge):
    case, iv, dv = problem(pkg, npv)
    rng = np.random.default_rng([npv, fwd, edge])
    for _ in range(200):
        yr, xr, yp, xp, ys, xs = step(L, iv, dv, fwd, edge, cells(pkg, rng, npv, case.params["pref"]), rng)
        assert np.array_equal(yr[:npv], yp[:npv])
        assert np.array_equal(xr[:npv], xp[:npv])
        assert np.abs(xr[:npv]).max() > 0.0


@pytest.mark.parametrize("npv", [7, 9])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e200])
def test_a_non_finite_operand_reaches_the_same_rows(L, pkg, npv, value):
    """A number of a cell or its neighbours that is not finite (or whose
    products overflow) leaves the rows finite that it leaves finite in the
    form without lanes; which of infinity and NaN the others hold may differ
    only where the energy row, and so the cell's temperature, is one of them."""
    case, iv, dv = problem(pkg, npv)
    for fwd in (0, 1):
        for item in range(42):
            for cell in range(4):
                rng = np.random.default_rng([npv, fwd, item, cell])
                c = cells(pkg, rng, npv, case.params["pref"])
                c[cell, item] = value
                yr, xr, _, _, ys, xs = step(L, iv, dv, fwd, cell & 1, c, rng)
                assert np.array_equal(np.isfinite(yr[:npv]), np.isfinite(ys[:npv])), (item, cell)
                assert np.array_equal(np.isfinite(xr[:npv]), np.isfinite(xs[:npv])), (item, cell)
                if not np.array_equal(np.isnan(xr[:npv]), np.isnan(xs[:npv])):
                    assert not np.isfinite(xr[4]), (item, cell)      # the cell's temperature is lost in either
