"""The shorter form of the face physics (harm_fast.h) against the general one
(harm_device.h), which the oracle tests pin: equal values wherever it holds,
and not held where a stencil or a flux is not finite.  Host build; the flux
kernels that run the two forms are compared on the GPU."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import harm_ramt_amd as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "fast_shim.cpp")
LIB = os.path.join(ROOT, "tests", "_shim", "fast_shim.so")
UP = [(0, 0), (0, 1), (0, 2), (0, 3), (1, 1), (1, 2), (1, 3), (2, 2), (2, 3), (3, 3)]


@pytest.fixture(scope="module")
def fast():
    src = [SRC] + [os.path.join(ROOT, "harm_ramt_amd", "csrc", f) for f in ("harm_fast.h", "harm_device.h")]
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(map(os.path.getmtime, src)):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.check_call([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O2",
                               "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", SRC, "-o", LIB])
    return ctypes.CDLL(LIB)


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)


def test_shared_reciprocal_is_the_ieee_quotient(fast):
    rng = np.random.default_rng(1)
    n = 400000
    with np.errstate(all="ignore"):
        a = rng.uniform(1, 2, n) * np.exp2(rng.integers(-1074, 1023, n).astype(float)) * rng.choice([-1, 1], n)
        d = rng.uniform(1, 2, n) * np.exp2(rng.choice([-1074, -1022, -100, -96, -95, -60, -1, 0, 1, 60, 64, 65, 66, 1022], n)
                                           .astype(float)) * rng.choice([-1, 1], n)
        special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, 1.7976931348623157e308, 1.0])
        k = rng.random(n) < 0.05
        a[k] = rng.choice(special, k.sum())
        k = rng.random(n) < 0.05
        d[k] = rng.choice(special, k.sum())
        want = a / d
    q = np.zeros(n)
    fast.shim_quotients(ctypes.c_long(n), _p(a), _p(d), _p(q))
    assert same(q, want)
    fin = ~np.isnan(want)
    assert np.array_equal(np.signbit(q[fin]), np.signbit(want[fin]))


def test_para4_edges(fast):
    rng = np.random.default_rng(2)
    n = 300000
    y = rng.uniform(-1, 1, (n, 5))
    y[: n // 4] = np.round(y[: n // 4] * 2) / 2                       # ties, flats, extrema
    y[n // 4: n // 2] *= 10.0 ** rng.uniform(-320, 300, (n // 4, 1))  # every magnitude
    y[n // 2: n // 2 + 20000] *= 10.0 ** rng.uniform(-320, 0, (20000, 5))
    bad = rng.choice(n, 3000, replace=False)
    y[bad, rng.integers(0, 5, 3000)] = rng.choice([np.nan, np.inf, -np.inf, 1e308, -1e308], 3000)
    gen, fst, ok = np.zeros((n, 2)), np.zeros((n, 2)), np.zeros(n, np.int32)
    fast.shim_para4(ctypes.c_long(n), _p(y), _p(gen), _p(fst), _p(ok))
    assert not ok[~np.isfinite(y).all(-1)].any()
    k = ok == 1
    assert k[np.abs(y).max(-1) < 1e150].all()
    assert same(gen[k], fst[k])


@pytest.mark.parametrize("dir", [1, 2])
@pytest.mark.parametrize("eom,flux", [(0, 1), (0, 0), (1, 0), (1, 1)])
def test_face_fluxes(fast, dir, eom, flux):
    rng = np.random.default_rng(10 * dir + 2 * eom + flux)
    g = H.grid_mks(24, 20)
    geom = H.Geometry(g)
    pos = dir - 1
    geo = np.stack([geom.gcov[:, :, pos, a, b] for a, b in UP] + [geom.gcon[:, :, pos, 0, m] for m in range(4)] +
                   [geom.gcon[:, :, pos, dir, dir], geom.gdet[:, :, pos]], -1).reshape(-1, 16)
    geo = np.ascontiguousarray(np.tile(geo, (40, 1)))
    n = len(geo)

    def states():
        p = np.zeros((n, 8))
        p[:, 0] = 10.0 ** rng.uniform(-8, 1, n)
        p[:, 1] = p[:, 0] * 10.0 ** rng.uniform(-6, 1, n)
        p[:, 2:5] = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-4, 0.7, (n, 1))
        p[:, 5:8] = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-3, 0, (n, 1))
        k = rng.random(n) < 0.3
        p[k, 5:8] *= 10.0 ** rng.uniform(-322, -30, (k.sum(), 1))   # fields next to nothing
        p[rng.random(n) < 0.1, 5:8] = 0.0
        p[rng.random(n) < 0.1, 2:5] = 0.0
        k = rng.random(n) < 0.05
        p[k, 1] *= -1                                               # failed inversions' energies
        if eom:
            p[:, :2] = 0.0
        return p
    pl, pr = states(), states()
    pr[: n // 3] = pl[: n // 3]
    bad = rng.choice(n, 500, replace=False)
    pl[bad, rng.integers(0, 8, 500)] = rng.choice([np.nan, np.inf, -np.inf, 1e300], 500)
    prm = np.array([4.0 / 3.0, eom, flux, 25.0, 4, 0.9, g.dx1, g.dx2])
    Fg, Ff, dg, df = np.zeros((n, 8)), np.zeros((n, 8)), np.zeros(n), np.zeros(n)
    fail, ok = np.zeros((n, 2), np.int32), np.zeros(n, np.int32)
    fast.shim_faces(_p(prm), dir, ctypes.c_long(n), _p(geo), _p(pl), _p(pr), _p(Fg), _p(dg), _p(Ff), _p(df), _p(fail),
                    _p(ok))
    k = ok == 1
    usual = np.ones(n, bool)
    usual[bad] = False
    finite = np.isfinite(Fg).all(-1)
    assert not k[~finite].any()
    moving = dg < 1e9   # some wave speed: a face without any takes the general form
    assert k[usual & finite & moving].mean() > 0.999
    assert same(Fg[k], Ff[k]) and same(dg[k], df[k])
    assert np.array_equal(fail[k, 0], fail[k, 1])


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2", [(4, 4), (5, 61), (6, 62), (7, 64), (11, 65), (33, 47)])
@pytest.mark.parametrize("scheme", [dict(lim=H.PARA), dict(lim=H.MC), dict(lim=H.PARA, fluxmethod=H.LAXFFLUX),
                                    dict(lim=H.MC, fluxmethod=H.LAXFFLUX, eomtype=H.EOMFFDE)])
def test_gpu_shared_fluxes_equal_the_general_kernel(n1, n2, scheme):
    """k_flux_shared against the thread-per-face kernel, on a state that holds
    zeros, fields down to the smallest numbers, velocities over gammamax,
    infinities and NaN."""
    g = H.grid_mks(n1, n2)
    geom = H.Geometry(g)
    rng = np.random.default_rng(n1 * 100 + n2)
    p = np.zeros((n1 + 6, n2 + 6, 8))
    p[..., 0] = 10.0 ** rng.uniform(-5, 0, p.shape[:2])
    p[..., 1] = p[..., 0] * 10.0 ** rng.uniform(-4, 0, p.shape[:2])
    p[..., 2:5] = rng.normal(size=p.shape[:2] + (3,)) * 0.1
    p[..., 5:8] = rng.normal(size=p.shape[:2] + (3,)) * 0.1 * 10.0 ** -(20.0 * np.arange(n1 + 6)[:, None, None] % 320)
    if "eomtype" in scheme:
        p[..., :2] = 0.0
    h = H.Harm(H.make_params(n1, n2, g.dx1, g.dx2, **scheme), geom)

    def fluxes(variant, state):
        h.set_array(H.P, state)
        h.set_array(H.F1, np.zeros_like(p))
        h.set_array(H.F2, np.zeros_like(p))
        h.set_tuning(variant, H.BOUND_KERNELS)
        dt = [h.fluxcalc(H.P, d) for d in (1, 2)]
        return h.get_array(H.F1), h.get_array(H.F2), dt

    def check(state):
        a, b = fluxes(H.FLUX_FACE_64x4, state), fluxes(H.FLUX_SHARED, state)
        assert same(a[0], b[0]) and same(a[1], b[1]) and a[2] == b[2]
        return a
    assert np.isfinite(check(p)[0]).all()
    q = p.copy()
    q[n1 // 2, n2 // 2, 2] = 300.0
    q[n1 // 2 + 3, n2 // 2 + 1, 5:8] = 0.0
    check(q)
    for v in (np.nan, np.inf, -np.inf, 1e308):
        for k in (0, 3, 6):
            q = p.copy()
            q[3 + n1 // 2, 3 + n2 // 3, k] = v
            check(q)
