"""The hand-written reverse passes of the adjoint (adjoint_point.hpp, compiled
for the host) against dual-number passes of the same templated physics: the
reconstruction under every limiter, the Roe and AUSM+-up flux cores, the
equation of state and the viscous flux, over states that reach the branches
of each.  Both differentiate the same operations and follow the same
selections, so they differ by rounding only: 1e-10 of the largest entry of a
gradient, 1e4 ulps for sums that cancel to as little as 1e-2 of their terms
over some hundred operations."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
TOL = 1e-10
# (normal, first, second transverse) offset of the face's 38 stencil points from its left cell
STENCIL = [(n, e, t) for t in (-1, 0, 1) for e in (-1, 0, 1) for n in (0, 1)] \
    + [(n, e, t) for n in (-1, 2) for t in (-1, 0, 1) for e in (-1, 0, 1)] + [(-2, 0, 0), (3, 0, 0)]


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("adjrev") / "libadjcheck.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-ffp-contract=off", "-std=c++17",
                    "-fPIC", "-shared", "-w", os.path.join(HERE, "native", "adjcheck.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def same(rev, dual, what):
    scale = np.max(np.abs(dual))
    assert np.all(np.isfinite(rev)) and np.max(np.abs(rev - dual)) <= TOL * scale, (what, rev, dual)


@pytest.mark.parametrize("mlp", [0, 1])
@pytest.mark.parametrize("nlim", range(11))
def test_reconstruction(L, nlim, mlp):
    rng = np.random.default_rng(10 * nlim + mlp)
    hit = 0
    for trial in range(1500):
        # a quadratic field (often close to an extremum, where the MLP bound is active) plus noise
        c = rng.standard_normal(5) * np.array([1.0, 0.5, 0.2, 0.2, 0.2])
        x = np.array([10.0 + c[0] * n + c[1] * n * n + c[2] * e + c[3] * t + c[4] * (e * e + t * t) for n, e, t in STENCIL])
        x += rng.standard_normal(38) * 10.0 ** rng.uniform(-3, 0)
        w = rng.standard_normal(2)
        rev, dual = np.zeros(38), np.zeros(38)
        L.ac_recon(nlim, mlp, dp(x), C.c_double(w[0]), C.c_double(w[1]), dp(rev), dp(dual))
        same(rev, dual, (trial, x))
        hit += np.any(dual[18:22] != 0) or np.any(dual[23:31] != 0) or np.any(dual[32:36] != 0) or np.any(dual[[0, 1, 4, 5, 12, 13, 16, 17]] != 0)
    if mlp and nlim in (2, 3, 4, 6, 7, 8):      # the limiters that read the bound: its extremum points were reached
        assert hit > 0


@pytest.mark.parametrize("bad", [0] + list(range(1, 37)))
def test_mlp_extrema_keep_the_order_of_a_comparison_chain(L, bad):
    """The extrema equal the chains (b < a) ? b : a over the points in order,
    also where point `bad` is a NaN: a chain that starts at it stays there, any
    other drops it."""
    rng = np.random.default_rng(bad)
    x, o = rng.standard_normal(38), np.zeros(10)
    if bad:
        x[bad - 1] = np.nan
    L.ac_extrema(dp(x), dp(o))
    chains = [range(1, 18, 2), range(2, 19, 2), range(1, 19), range(19, 28), range(28, 37)]
    for c, ll in enumerate(chains):
        lo = hi = x[ll[0] - 1]
        for q in ll:
            lo = x[q - 1] if x[q - 1] < lo else lo
            hi = x[q - 1] if x[q - 1] > hi else hi
        assert np.array_equal([lo, hi], o[2 * c:2 * c + 2], equal_nan=True), (bad, c)


@pytest.mark.parametrize("npv", [7, 9])
@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("scheme", [1, 4])
def test_flux_core(L, scheme, prec, npv):
    rng = np.random.default_rng(100 * scheme + 10 * prec + npv)
    for trial in range(300):
        z = np.zeros(24)
        fast = trial % 3                        # low Mach, near u_ref, supersonic (low sound speed)
        for o in (0, 9):
            z[o] = rng.uniform(-3e4, 3e4)
            z[o + 1:o + 4] = rng.standard_normal(3) * (1.0, 12.0, 400.0)[fast]
            z[o + 4] = rng.uniform(290, 310)
            z[o + 5:o + 7] = rng.uniform(0, 0.1, 2)
            if npv == 9:
                z[o + 7], z[o + 8] = rng.uniform(0, 1), rng.uniform(1, 1e4)
        z[18], z[20] = rng.uniform(1, 1000, 2)
        z[19], z[21] = rng.uniform(1e5, 3e5, 2)
        z[22] = (1450.0, 40.0, 90.0)[fast] ** 2 * rng.uniform(0.5, 2)
        z[23] = 10.0
        n3 = rng.standard_normal(3) * 1e-3
        g = np.zeros(9)
        g[:npv] = rng.standard_normal(npv) / np.array([1, 10, 10, 10, 1e5, 1, 1, 1, 1])[:npv]
        rev, dual = np.zeros(24), np.zeros(24)
        L.ac_flux(scheme, prec, npv, C.c_double(4.3e4), C.c_double(20.0), dp(n3), dp(z), dp(g), dp(rev), dp(dual))
        # each input on its own scale: the change its own size makes
        ref = np.maximum(np.abs(z), 1e-3)
        same(rev * ref, dual * ref, (trial, z))


@pytest.mark.parametrize("c2", [0, 1])
def test_equation_of_state(L, c2):
    rng = np.random.default_rng(5 + c2)
    for trial in range(300):
        x4 = np.array([10.0 ** rng.uniform(2.0, 6.5), rng.uniform(276, 480), rng.choice([0.0, 1e-9, rng.uniform(0, 1)]), 0.0])
        x4[3] = rng.choice([0.0, rng.uniform(0, 1 - x4[2])])
        w = np.zeros(13)
        # one property at a time: their sizes differ by many orders
        m = 2 if c2 else trial % 13
        w[m] = 1.0
        rev, dual = np.zeros(4), np.zeros(4)
        L.ac_eos(1, c2, dp(x4), dp(w), dp(rev), dp(dual))
        ref = np.maximum(np.abs(x4), 1e-3)
        if not np.any(dual):
            assert not np.any(rev)
            continue
        same(rev * ref, dual * ref, (trial, m, x4))


@pytest.mark.parametrize("iturb", [-2, 0])
def test_viscous_flux(L, iturb):
    rng = np.random.default_rng(7 - iturb)
    for trial in range(300):
        met = np.concatenate([rng.standard_normal(27) * 1e-4, [1e-7, 10.0 ** rng.uniform(-6, -2), 1.2e-7, 10.0 ** rng.uniform(-6, -2)]])
        z = np.zeros(33)
        z[:18] = rng.standard_normal(18)
        z[15:18] *= 10.0 ** rng.uniform(0, 3)
        z[18:21] = rng.standard_normal(3) * 10
        z[21], z[22] = rng.choice([0.0, 10.0 ** rng.uniform(-6, 0)]), 10.0 ** rng.uniform(0, 5)
        z[23:27:2] = rng.uniform(5e-4, 1.5e-3, 2)
        z[24:27:2] = rng.uniform(0.5, 0.7, 2)
        z[27:29] = rng.uniform(4e3, 4.3e3, 2)
        z[29:31] = rng.uniform(1, 1000, 2)
        z[31:33] = 10.0 ** rng.uniform(-4, -1, 2)
        g = rng.standard_normal(9) / np.array([1, 10, 10, 10, 1e5, 1, 1, 1, 1])
        rev, dual = np.zeros(33), np.zeros(33)
        L.ac_visc(iturb, dp(met), dp(z), dp(g), dp(rev), dp(dual))
        ref = np.maximum(np.abs(z), 1e-12)
        ref[21] = max(ref[21], 1e-6)
        same(rev * ref, dual * ref, (trial, z))
