"""Kernels compiled for a geometry pattern (entries that hold one value over
all zones are read from zone 0) against the oracle, to the bit: tables that
have the pattern, tables that break it in the last zone of one entry, and a
context and a batch whose tables change from one to the other between steps.
"""
import numpy as np
import pytest

import harm_ramt_amd as H
from tests.helpers import problem, same
from tests.test_gpu_parity import gpu_ctx, oracle_ctx

pytestmark = pytest.mark.gpu
NG = 3


def broken(geom, n1, n2):
    """the tables with one more value in entries that hold one: g_{t theta} at
    the centre and g^{t theta} at the x1 face of an interior zone, the
    connection's Gamma^theta_{t theta}, and on a uniform grid with them gdet at
    a corner"""
    gcov, gcon, gdet, conn, floors = [np.array(x) for x in geom.tables()]
    i, j = NG + n1 - 1, NG + n2 - 2
    gcov[i, j, 3, 0, 2] = gcov[i, j, 3, 2, 0] = 1e-3
    gcon[i, j, 0, 0, 2] = gcon[i, j, 0, 2, 0] = 2e-3
    conn[i, j, 2, 0, 2] = conn[i, j, 2, 2, 0] = 3e-3
    if np.all(gdet == gdet[0, 0, 0]):
        gdet[i, j, 2] *= 1.001
    return gcov, gcon, gdet, conn, floors


@pytest.mark.parametrize("kind,n1,n2,lim", [("ks", 17, 40, H.PARA), ("ks", 160, 230, H.PARA), ("ks", 160, 230, H.VANL),
                                            ("mink", 24, 33, H.MC), ("mink", 160, 230, H.MC), ("mink", 24, 33, H.PARA),
                                            ("ffde", 32, 48, H.MC), ("ffde", 160, 230, H.MC)])
def test_geometry_patterns(kind, n1, n2, lim):
    print(f"[case] geometry patterns: {kind} {n1}x{n2} lim={lim}", flush=True)
    flux = H.LAXFFLUX if kind == "ffde" else H.HLLFLUX
    g, geom, p0, prm = problem(kind, n1, n2, lim=lim, fluxmethod=flux, timeorder=2)
    plain, other = geom.tables(), broken(geom, n1, n2)
    dt0 = 1e-4 if kind == "mink" else 1e-3
    a, o = gpu_ctx(geom, prm, p0, dt0), oracle_ctx(geom, prm, p0, dt0)
    a.set_tuning(H.FLUX_SHARED, H.BOUND_INUPDATE)
    runs = [gpu_ctx(geom, prm, p0, dt0) for _ in range(2)]
    b = H.Batch(runs)
    for k, tables in enumerate((plain, other, plain)):
        if k:
            for h in (a, runs[1]):
                h.set_geometry(*tables)
            o.set_geometry(*tables)
            if k == 1:
                still = runs[0].get_array(H.P)
        a.step_ch()
        a.step_n(2)
        b.step_n(3)
        for _ in range(3):
            o.step()
        assert a.get_time() == o.get_time() == runs[1].get_time()
        assert same(a.get_array(H.P), o.get_array(0)), f"tables {k}"
        assert same(runs[1].get_array(H.P), o.get_array(0)), f"tables {k}: batch"
        if k == 0:
            assert same(runs[0].get_array(H.P), o.get_array(0))
    assert not same(still, runs[0].get_array(H.P))
    b.close()
