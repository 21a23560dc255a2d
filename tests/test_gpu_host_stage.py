"""Inversions of zones held on the host by way of the context's pinned staging:
the same solutions whatever the number of zones is (one, either side of the
staging's sizes, and past its bound, where the call allocates for itself), and
with two threads on one context."""
import threading

import numpy as np
import pytest

import harm_ramt_amd as H
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
N1, N2, MOST = 16, 24, 1 << 16


@pytest.fixture(scope="module")
def inversion():
    g = H.grid_mks(N1, N2)
    geom = H.Geometry(g)
    prm = H.make_params(N1, N2, g.dx1, g.dx2)
    h, o = H.Harm(prm, geom), Oracle(H.params_dict(prm))
    o.set_geometry(*geom.tables())
    rng = np.random.default_rng(5)
    zones = np.stack([rng.integers(-3, N1 + 3, 600), rng.integers(-3, N2 + 3, 600)], axis=1).astype(np.int32)
    U, guess = np.zeros((600, 8)), np.zeros((600, 8))
    for t, (i, j) in enumerate(zones):
        rho = 10 ** rng.uniform(-4, 0)
        pr = np.array([rho, rho * 10 ** rng.uniform(-3, 1), *rng.normal(0, 1, 3), *(rng.normal(0, 0.3, 3) * np.sqrt(rho))])
        U[t] = o.primtoU(int(i), int(j), 3, pr)
        guess[t] = pr * (1 + rng.normal(0, 0.05, 8))
    want = [h.utoprimgen(zones[t:t + 1], U[t:t + 1], guess[t:t + 1]) for t in range(600)]
    return h, zones, U, guess, np.concatenate([w[0] for w in want]), np.concatenate([w[1] for w in want])


@pytest.mark.parametrize("n", [MOST + 1, MOST, 257, 256, 255, 65, 1])
def test_every_size_gives_the_zones_solutions(inversion, n):
    h, zones, U, guess, pr, flag = inversion
    k = np.random.default_rng(n).integers(0, 600, n)
    a, f = h.utoprimgen(zones[k], U[k], guess[k])
    assert a.tobytes() == pr[k].tobytes() and np.array_equal(f, flag[k])


def test_two_threads_on_one_context(inversion):
    h, zones, U, guess, pr, flag = inversion
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for n in (300, 700, 40, 2000):
            k = rng.integers(0, 600, n)
            a, f = h.utoprimgen(zones[k], U[k], guess[k])
            if a.tobytes() != pr[k].tobytes() or not np.array_equal(f, flag[k]):
                bad.append((seed, n))
    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
