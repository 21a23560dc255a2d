"""The serial sums of the accounting formed by runs (harm_chain.h): the same bits
as the additions one by one, for terms that tie, cancel, cross binades, vanish
or are not finite.  The maps are checked on the host, the sums that the GPU
forms with them on the GPU."""
import ctypes
import os

import numpy as np
import pytest

import harm_ramt_amd as H
from tests.test_fast_math import _p, fast  # noqa: F401  (the host build)


def plain(t, s):
    with np.errstate(all="ignore"):
        return np.add.accumulate(np.concatenate([[s], t]))[-1]


def terms(kind, rng, n):
    x = rng.standard_normal(n)
    if kind == "positive":
        return np.abs(x)
    if kind == "cancelling":
        return x
    if kind == "ties":  # few bits: sums end on half a unit of the last place all the time
        return rng.integers(-8, 24, n) * 2.0 ** -53
    if kind == "wide":
        return x * np.exp2(rng.integers(-80, 20, n).astype(float))
    if kind == "drift":
        return 1e-4 * (x + 0.3)
    if kind == "sparse":
        return np.where(rng.random(n) < 0.01, x, np.where(rng.random(n) < 0.5, 0.0, -0.0))
    if kind == "special":
        t = x.copy()
        k = rng.random(n) < 2e-4
        t[k] = rng.choice([np.inf, -np.inf, np.nan, 5e-324, 1.7e308, -1.7e308], k.sum())
        return t
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["positive", "cancelling", "ties", "wide", "drift", "sparse", "special"])
def test_runs_give_the_serial_sum(fast, kind):  # noqa: F811
    rng = np.random.default_rng(sum(map(ord, kind)))
    fast.shim_chain.restype = ctypes.c_double
    held = ctypes.c_long()
    total = 0
    for start in [0.0, 1.0, 1.0 + 2.0 ** -52, -1.0, -(2.0 - 2.0 ** -52), 3.7e5, -2.5e-9, 1e-300, 1e300, 5e-324]:
        for n in (16, 1024, 16 * 1000):
            t = terms(kind, rng, n) * rng.choice([1.0, 1.0, -1.0, 1e-3])
            got = fast.shim_chain(ctypes.c_long(n), _p(t), ctypes.c_double(start), ctypes.byref(held))
            want = plain(t, start)
            assert np.float64(got).tobytes() == np.float64(want).tobytes() or (np.isnan(got) and np.isnan(want))
            total += held.value
    if kind != "special":
        assert total > 300  # the maps hold for most runs


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2", [(16, 32), (33, 70), (128, 129)])
def test_source_sums_on_the_gpu(n1, n2):
    """sourceadd over many steps: the ordered sums against the oracle's loop."""
    from oracle.oracle import Oracle

    g = H.grid_mks(n1, n2)
    geom = H.Geometry(g)
    p0 = H.init_fishmon(geom)
    prm = H.make_params(n1, n2, g.dx1, g.dx2)
    h, o = H.Harm(prm, geom), Oracle(H.params_dict(prm))
    o.set_geometry(*geom.tables())
    regions = H.ener_regions(g)
    h.set_array(H.P, p0)
    h.bound_prim(H.P)
    o.set_array(0, p0)
    o.bound_prim(0)
    for m in (h, o):
        m.set_time(0.0, 1e-3, 1e30)
        m.acct_setup(*regions)
    for _ in range(4):
        h.step_ch()
        o.step()
    a, b = h.acct(), o.acct()
    for name in ("sourceadd", "fladd", "fladdterms", "pdot", "pcum", "pdotterms", "pdottermsjet2", "frdot", "lumvsr"):
        assert np.array_equal(np.asarray(a[name]), np.asarray(b[name])), name
