"""The substage in one launch (fluxes and update of an 8 x 8 tile by one
workgroup) against the oracle and, bit for bit, against the same step in two
launches, at tile edges and remainders, with every compiled scheme.  Chosen for
grids of at most 512 tiles; the last case lies one column of tiles past that
line.  The bar is equality: the tiles call the functions of the two launches in
their order.
"""
import numpy as np
import pytest

import harm_ramt_amd as H
from tests.helpers import problem, same
from tests.test_gpu_parity import bits, gpu_ctx, oracle_ctx, strong_field_at_edges

pytestmark = pytest.mark.gpu
NG = 3

CASES = [("ks", 8, 8, H.PARA, 4), ("ks", 9, 16, H.PARA, 4), ("ks", 4, 33, H.PARA, 3), ("ks", 17, 7, H.PARA, 2),
         ("ks", 33, 47, H.MC, 4), ("ks", 32, 64, H.VANL, 4), ("ks", 24, 24, H.PARA, 1), ("mink", 15, 23, H.MC, 4),
         ("mink", 7, 40, H.PARA, 2), ("ffde", 17, 34, H.MC, 2), ("ks", 128, 256, H.PARA, 4), ("ks", 128, 257, H.PARA, 4)]


@pytest.mark.parametrize("kind,n1,n2,lim,order", CASES)
def test_one_launch_substage(kind, n1, n2, lim, order):
    print(f"[case] one-launch substage: {kind} {n1}x{n2} lim={lim} order={order}, 14 steps", flush=True)
    flux = H.LAXFFLUX if kind == "ffde" else H.HLLFLUX
    g, geom, p0, prm = problem(kind, n1, n2, lim=lim, fluxmethod=flux, timeorder=order)
    p0 = p0.copy()
    if kind == "ks" and n1 > 4 and n2 > 8:
        strong_field_at_edges(p0, n1, n2)
    dt0 = 1e-4 if kind == "mink" else 1e-3
    a, b, o = gpu_ctx(geom, prm, p0, dt0), gpu_ctx(geom, prm, p0, dt0), oracle_ctx(geom, prm, p0, dt0)
    a.set_tuning(H.FLUX_SHARED, H.BOUND_INUPDATE)
    b.set_tuning(H.FLUX_SHARED, H.BOUND_FUSED)  # two launches, and the fill its own
    for s in range(14):
        a.step_ch()
        b.step_ch()
        o.step()
        what = f"step {s + 1}"
        assert a.get_time() == o.get_time() == b.get_time(), what
        pa = a.get_array(H.P)
        assert same(pa, o.get_array(0)), what + ": state vs oracle"
        assert np.array_equal(bits(pa), bits(b.get_array(H.P))), what + ": bits vs two launches"
        assert np.array_equal(a.get_pflag(), b.get_pflag()), what + ": flags"
        _same_fluxes(a, b, n1, n2, what)
    assert a.nstroke() == o.nstroke() == b.nstroke()
    assert a.failures() == b.failures() and a.failures()[1] == o.failed()


def _same_fluxes(a, b, n1, n2, what):
    """the fluxes a step leaves: x1 faces i in [0,N1], j in [-1,N2], x2 faces
    i in [-1,N1], j in [0,N2]"""
    for sel, w in ((H.F1, np.s_[NG:NG + n1 + 1, NG - 1:NG + n2 + 1]), (H.F2, np.s_[NG - 1:NG + n1 + 1, NG:NG + n2 + 1])):
        assert np.array_equal(bits(a.get_array(sel)[w]), bits(b.get_array(sel)[w])), what + ": fluxes"


BATCHES = {  # runs (kind, n1, n2, order): one scheme or several, below and above 512 tiles together
    "tori": [("ks", 33, 47, 4), ("ks", 64, 60, 4), ("ks", 4, 9, 4)],
    "tori_large": [("ks", 117, 160, 4), ("ks", 120, 163, 4)],
    "vortices": [("mink", 15, 23, 2), ("mink", 32, 32, 2)],
    "vortices_large": [("mink", 170, 200, 4)],
    "mixed_large": [("mink", 130, 161, 2), ("ks", 101, 131, 2), ("ffde", 16, 30, 2)],
    "first_order": [("ks", 24, 24, 1), ("ks", 17, 66, 1)],
}


@pytest.mark.parametrize("case", sorted(BATCHES))
def test_batch_with_the_fill_in_the_update(case):
    """Every run of a batch against the same run alone with the fills in
    launches of their own: state, flags, fluxes, time, counts."""
    print(f"[case] batch {case}: {BATCHES[case]}, 12 steps", flush=True)
    runs, alone = [], []
    for kind, n1, n2, order in BATCHES[case]:
        flux = H.LAXFFLUX if kind == "ffde" else H.HLLFLUX
        lim = H.PARA if kind == "ks" else H.MC
        g, geom, p0, prm = problem(kind, n1, n2, lim=lim, fluxmethod=flux, timeorder=order)
        p0 = p0.copy()
        if kind == "ks" and n1 > 4:
            strong_field_at_edges(p0, n1, n2)
        for out in (runs, alone):
            out.append(gpu_ctx(geom, prm, p0, 1e-4 if kind == "mink" else 1e-3))
        alone[-1].set_tuning(H.FLUX_SHARED, H.BOUND_FUSED)
    b = H.Batch(runs)
    for n in (1, 11):
        b.step_n(n)
        for k, (x, y) in enumerate(zip(runs, alone)):
            y.step_n(n)
            what = f"run {k}"
            assert x.get_time() == y.get_time(), what
            assert np.array_equal(bits(x.get_array(H.P)), bits(y.get_array(H.P))), what + ": state"
            assert np.array_equal(x.get_pflag(), y.get_pflag()), what + ": flags"
            assert x.nstroke() == y.nstroke() and x.failures() == y.failures(), what
            _same_fluxes(x, y, *BATCHES[case][k][1:3], what)
    b.close()
