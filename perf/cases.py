"""The work that users of this framework have it do, as measurable cases.

A case is one pass through the public entry points of ``harm_ramt_amd``:

steps       a context stepped on: ``step_ch()`` (one call a step, the form of
            the reference's main loop) or ``step_n(k)`` (k steps between dumps),
            then the time read back.  The Fishbone-Moncrief torus (GRMHD,
            outflow and polar sides), the Orszag-Tang vortex (GRMHD, periodic,
            Minkowski) and the force-free split monopole, over the limiters,
            flux methods and Runge-Kutta orders that the runs use.
accounting  torus steps with the conservation accounting on, and its
            accumulators read, as before an energy log line.
batch       several tori of different sizes and spins advanced together.
adjoint     a forward run from a given state, the magnetic energy, and the
            gradient with respect to that state.
invert      Utoprimgen of a list of zones held on the host.

Every state continues where its last pass left it, as a run does; an adjoint
or an inversion starts from its own inputs each time.
"""
import functools
import math
import random

import numpy as np
import torch

import harm_ramt_amd as H

NG = 3
LIMS = {"mc": H.MC, "para": H.PARA, "vanl": H.VANL, "minm": H.MINM}
FLUXES = {"hll": H.HLLFLUX, "laxf": H.LAXFFLUX}
SUBSTEPS = {2: 2, 3: 3, 4: 4}


def listed():
    return [
        # the reference's main loop: one call a step, on the size of a quick look; launches and latency count
        {"name": "torus_32x64_one_step", "do": "steps", "problem": "torus", "n1": 32, "n2": 64, "lim": "para",
         "flux": "hll", "order": 4, "steps": 1, "call": "step_ch"},
        # a small production grid whose sides fill no tile of any kernel
        {"name": "torus_97x131", "do": "steps", "problem": "torus", "n1": 97, "n2": 131, "lim": "para",
         "flux": "hll", "order": 4, "steps": 16, "call": "step_n"},
        # the headline run of the benchmark, between two dumps
        {"name": "torus_256", "do": "steps", "problem": "torus", "n1": 256, "n2": 256, "lim": "para",
         "flux": "hll", "order": 4, "steps": 20, "call": "step_n"},
        # the torus on a fine grid
        {"name": "torus_512", "do": "steps", "problem": "torus", "n1": 512, "n2": 512, "lim": "para",
         "flux": "hll", "order": 4, "steps": 10, "call": "step_n"},
        # Orszag-Tang vortex: periodic, MC slopes, the setting of the gradient runs
        {"name": "orszag_tang_256", "do": "steps", "problem": "orszag_tang", "n1": 256, "n2": 256, "lim": "mc",
         "flux": "hll", "order": 4, "steps": 16, "call": "step_n"},
        # force-free magnetosphere at the size of the spin scan
        {"name": "monopole_512", "do": "steps", "problem": "monopole", "n1": 512, "n2": 512, "lim": "mc",
         "flux": "laxf", "order": 2, "steps": 16, "call": "step_n"},
        # a torus run that logs its conserved totals
        {"name": "accounting_256", "do": "accounting", "problem": "torus", "n1": 256, "n2": 256, "lim": "para",
         "flux": "hll", "order": 4, "steps": 4, "tree": False},
        # a parameter scan: tori of several sizes and spins in one batch
        {"name": "batch_12_tori", "do": "batch", "runs": 12, "draw": 2024, "steps": 4},
        # a gradient of an Orszag-Tang run, every substage's state kept
        {"name": "gradient_128", "do": "adjoint", "problem": "orszag_tang", "n1": 128, "n2": 128, "lim": "mc",
         "flux": "hll", "order": 4, "steps": 32, "every": 32},
        # conserved to primitive for zones that a host program holds
        {"name": "invert_4096", "do": "invert", "problem": "torus", "n1": 64, "n2": 64, "zones": 4096},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["steps", "steps", "steps", "steps", "steps", "accounting", "batch", "adjoint", "invert"])
    if do == "batch":
        return {"do": "batch", "runs": rng.randint(3, 12), "draw": rng.randrange(1 << 20), "steps": rng.randint(1, 4)}
    if do == "adjoint":
        steps = rng.randint(6, 32)
        return {"do": do, "problem": "orszag_tang", "n1": _spread(rng, 24, 160), "n2": _spread(rng, 24, 160),
                "lim": rng.choice(["mc", "mc", "vanl", "minm"]), "flux": rng.choice(["hll", "laxf"]),
                "order": rng.choice([2, 4, 4]), "steps": steps, "every": rng.choice([steps, 5])}
    if do == "invert":
        return {"do": do, "problem": "torus", "n1": _spread(rng, 24, 128), "n2": _spread(rng, 24, 128),
                "zones": _spread(rng, 100, 16000)}
    if do == "accounting":
        return {"do": do, "problem": "torus", "n1": _spread(rng, 32, 256), "n2": _spread(rng, 32, 256),
                "lim": "para", "flux": "hll", "order": rng.choice([2, 4]), "steps": rng.randint(1, 4),
                "tree": rng.choice([False, True])}
    problem = rng.choice(["torus", "torus", "torus", "orszag_tang", "monopole"])
    n1, n2 = _spread(rng, 24, 512), _spread(rng, 24, 512)
    call = rng.choice(["step_n", "step_n", "step_n", "step_ch"])
    if problem == "monopole":
        lim, flux, order = rng.choice(["mc", "mc", "para"]), rng.choice(["laxf", "hll"]), rng.choice([2, 2, 4])
    else:
        lim = rng.choice(["para", "para", "mc"] if problem == "torus" else ["mc", "mc", "para", "vanl"])
        flux, order = rng.choice(["hll", "hll", "laxf"]), rng.choice([4, 4, 3, 2])
    steps = 1 if call == "step_ch" else rng.randint(4, 20)
    steps = max(1, min(steps, 10 * 512 * 512 // (n1 * n2)))
    return {"do": do, "problem": problem, "n1": n1, "n2": n2, "lim": lim, "flux": flux, "order": order,
            "steps": steps, "call": call}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _geometry(problem, n1, n2, a):
    """The grid's tables, which a run reads once and keeps: the same for every seed."""
    if problem == "orszag_tang":
        return H.Geometry(H.grid_cartesian(n1, n2))
    if problem == "monopole":
        return H.Geometry(H.grid_mks(n1, n2, a=a, Rout=100.0, hslope=0.1))
    return H.Geometry(H.grid_mks(n1, n2, a=a, Rout=40.0, hslope=0.3))


def _spin(problem):
    return {"torus": 0.9375, "monopole": 0.9, "orszag_tang": 0.0}[problem]


def _params(problem, geom, lim, flux, order):
    g = geom.grid
    kw = dict(lim=LIMS[lim], fluxmethod=FLUXES[flux], timeorder=order)
    if problem == "orszag_tang":
        kw.update(gam=5.0 / 3.0, cour=0.8, bc=(H.PERIODIC,) * 4, fixupflux=0, poledeath=0)
    elif problem == "monopole":
        kw.update(eomtype=H.EOMFFDE, poledeath=0)
    return H.make_params(g.n1, g.n2, g.dx1, g.dx2, **kw)


def _state(problem, geom, seed, rmax=12.0, beta=100.0):
    rng = np.random.default_rng(seed)
    if problem == "torus":  # 4 % perturbations of u
        return H.init_fishmon(geom, rmax=rmax, beta=beta, randfact=4e-2, seed=int(rng.integers(1, 1 << 31)))
    if problem == "monopole":
        return H.init_monopole(geom, B0=float(rng.uniform(0.5, 2.0)))
    p = H.init_orszag_tang(geom)
    p[..., 0] *= 1.0 + 1e-2 * rng.uniform(-1, 1, p.shape[:2])
    p[..., 2:5] += 1e-3 * rng.uniform(-1, 1, p.shape[:2] + (3,))
    return p


FIRST_DT = {"torus": 1e-3, "monopole": 1e-3, "orszag_tang": 1e-3}


def _begin(h, p0, problem):
    h.set_array(H.P, p0)
    h.bound_prim(H.P)
    h.set_time(0.0, FIRST_DT[problem], 1e30)


def _context(problem, geom, p0, lim, flux, order):
    """A context at the start of its run; its kernels chosen, its graphs recorded."""
    h = H.Harm(_params(problem, geom, lim, flux, order), geom)
    _begin(h, p0, problem)
    return h


class _Device:
    """A context's state where it lies.  A tensor made of it holds this object, and so the context that owns the memory."""

    def __init__(self, h):
        self.owner = h
        self.__cuda_array_interface__ = {"shape": h.shape, "typestr": "<f8", "data": (h.array_ptr(H.P), False), "version": 3}


def _view(h):
    return torch.as_tensor(_Device(h), device="cuda")


def _tori(case):
    rng = random.Random(case["draw"])
    return [{"n1": 8 * rng.randint(6, 32) + rng.choice([0, 0, 0, 1, 5]), "n2": 8 * rng.randint(6, 32) + rng.choice([0, 0, 0, 3]),
             "a": round(rng.uniform(0.0, 0.95), 2), "rmax": rng.uniform(10, 16), "beta": rng.uniform(30, 300)}
            for _ in range(case["runs"])]


def _torus_states(case, seed):
    out = []
    for k, d in enumerate(_tori(case)):
        geom = _geometry("torus", d["n1"], d["n2"], d["a"])
        out.append((geom, _state("torus", geom, 1000 * seed + k, d["rmax"], d["beta"])))
    return out


def _inversion_inputs(case, seed):
    """Zones, U and guesses: the torus's zones, moved a little, as an evolved state's are."""
    geom = _geometry("torus", case["n1"], case["n2"], _spin("torus"))
    p = _state("torus", geom, seed)
    rng = np.random.default_rng(seed + 17)
    n = case["zones"]
    zones = np.stack([rng.integers(0, case["n1"], n), rng.integers(0, case["n2"], n)], -1).astype(np.int32)
    i, j = zones[:, 0] + NG, zones[:, 1] + NG
    pr = p[i, j].copy()
    pr[:, 0] = np.maximum(pr[:, 0], geom.floors[i, j, 0])
    pr[:, 1] = np.maximum(pr[:, 1], 1e-2 * pr[:, 0])
    pr[:, :2] *= np.exp(rng.uniform(-0.1, 0.1, (n, 2)))
    pr[:, 2:5] += rng.uniform(-1, 1, (n, 3)) * np.array([2e-2, 2e-3, 2e-3])
    pr[:, 5:8] += rng.uniform(-1, 1, (n, 3)) * (1e-2 * np.sqrt(pr[:, :1]) * np.array([1.0, 0.1, 0.1]))
    R = _Exact(geom.gcov[i, j], geom.gcon[i, j], geom.gdet[i, j], geom.conn[i, j], geom.floors[i, j], None, "cpu")
    t = torch.from_numpy(pr)
    U = R.flux(t, R.state(t, 3), 0, 3).numpy()
    guess = pr.copy()
    guess[:, :2] *= np.exp(rng.uniform(-0.05, 0.05, (n, 2)))
    guess[:, 2:5] += rng.uniform(-1, 1, (n, 3)) * 1e-3
    return geom, zones, U, guess, pr


def prepare(case, seed):
    do = case["do"]
    if do == "batch":
        runs = [_context("torus", geom, p0, "para", "hll", 4) for geom, p0 in _torus_states(case, seed)]
        batch = H.Batch(runs)
        batch.step_n(1)  # its kernels chosen, its graph recorded; then the run's start
        for h, (geom, p0) in zip(runs, _torus_states(case, seed)):
            _begin(h, p0, "torus")
        return {"case": case, "runs": runs, "batch": batch, "views": [_view(h) for h in runs]}
    if do == "invert":
        geom, zones, U, guess, _ = _inversion_inputs(case, seed)
        h = H.Harm(_params("torus", geom, "para", "hll", 4), geom)
        return {"case": case, "h": h, "zones": zones, "U": U, "guess": guess}
    problem = case["problem"]
    geom = _geometry(problem, case["n1"], case["n2"], _spin(problem))
    p0 = _state(problem, geom, seed)
    h = _context(problem, geom, p0, case["lim"], case["flux"], case["order"])
    s = {"case": case, "h": h, "p0": p0}
    if do == "adjoint":
        s["adjoint"] = H.Adjoint(h, case["steps"], case["every"])
        _gradient(s)
        return s
    # the first call chooses the kernels and records the graphs; then the run's start
    (h.step_ch if case.get("call") == "step_ch" else lambda: h.step_n(case["steps"]))()
    _begin(h, p0, problem)
    if do == "accounting":
        h.acct_setup(*H.ener_regions(geom.grid))
        if case["tree"]:
            h.acct_set_order(H.ACCT_TREE)
    s["view"] = _view(h)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _gradient(s):
    h, a = s["h"], s["adjoint"]
    _begin(h, s["p0"], s["case"]["problem"])
    a.forward()
    energy = a.seed_magnetic_energy()
    return {"energy": energy, "gradient": a.backward(), "dts": a.dts()}


def run(s):
    case = s["case"]
    do = case["do"]
    if do == "batch":
        s["batch"].step_n(case["steps"])
        return {"p": s["views"], "time": np.array([h.get_time() for h in s["runs"]])}
    if do == "adjoint":
        return _gradient(s)
    h = s["h"]
    if do == "invert":
        pr, flag = h.utoprimgen(s["zones"], s["U"], s["guess"])
        return {"pr": pr, "flag": flag}
    if case.get("call") == "step_ch":
        for _ in range(case["steps"]):
            h.step_ch()
    else:
        h.step_n(case["steps"])
    out = {"p": s["view"], "time": np.array(h.get_time())}
    if do == "accounting":
        out["acct"] = h.acct()
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# Bytes of one zone and substage: pi, pb read and pf written (192), the
# accumulated conserved state read and written (128), the geometry of its
# centre (30 numbers), its two faces (16 each) and its connection (40), read.
# Operations of one zone and substage: two faces (two reconstructed states,
# F, U and speeds of each, 8 components combined) about 4300; the update
# (U, source contraction, divergence, five Newton iterations) about 2400,
# and without the Newton iterations about 1700.
SUBSTAGE_BYTES = 192 + 128 + 8 * (30 + 2 * 16 + 40)
SUBSTAGE_FLOPS = {"torus": 6700, "orszag_tang": 6300, "monopole": 5500}


def work(case):
    do = case["do"]
    if do == "invert":  # the zone's indices, its U and guess in, its state and flag out, its metric
        return {"bytes": case["zones"] * (8 + 64 + 64 + 64 + 4 + 8 * 27), "flops": case["zones"] * 1000}
    if do == "batch":
        n = sum(d["n1"] * d["n2"] for d in _tori(case)) * case["steps"] * 4
        return {"bytes": n * SUBSTAGE_BYTES, "flops": n * SUBSTAGE_FLOPS["torus"]}
    n = case["n1"] * case["n2"] * case["steps"] * SUBSTEPS[case["order"]]
    w = {"bytes": n * SUBSTAGE_BYTES, "flops": n * SUBSTAGE_FLOPS[case["problem"]]}
    if do == "adjoint":  # the run, and its reverse: each operation's adjoint is about two
        w = {k: 3 * v for k, v in w.items()}
    return w


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
class _Exact:
    """The step written from its equations, on whole arrays: geometry at
    position 0 (x1 face), 1 (x2 face), 2 (corner), 3 (centre) of each zone."""

    def __init__(self, gcov, gcon, gdet, conn, floors, prm, dev):
        def put(x):
            return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device=dev)
        self.gcov, self.gcon, self.gdet, self.conn, self.floors = (put(x) for x in (gcov, gcon, gdet, conn, floors))
        self.prm, self.dev = prm, dev
        self.ffde = prm is not None and prm.eomtype == H.EOMFFDE
        self.gam = prm.gam if prm is not None else 4.0 / 3.0

    def geo(self, pos, at=None):
        g = (self.gcov[..., pos, :, :], self.gcon[..., pos, :, :], self.gdet[..., pos])
        return g if at is None else tuple(x[at] for x in g)

    # -- the zone's state, conserved quantities and fluxes --
    def gamma(self, p, g):
        u = p[..., 2:5]
        return torch.sqrt(1 + (u[..., :, None] * u[..., None, :] * g[0][..., 1:, 1:]).sum((-1, -2)))

    def limit(self, p, g, most):
        gam = self.gamma(p, g)
        f = torch.sqrt((most * most - 1) / torch.clamp(gam * gam - 1, min=1e-300))
        f = torch.where(gam > most, f, torch.ones_like(f))
        return torch.cat([p[..., :2], p[..., 2:5] * f[..., None], p[..., 5:]], -1)

    def state(self, p, pos, at=None):
        g = self.geo(pos, at)
        alpha = 1 / torch.sqrt(-g[1][..., 0, 0])
        gam = self.gamma(p, g)
        u0 = gam / alpha
        ui = p[..., 2:5] - (gam * alpha)[..., None] * g[1][..., 0, 1:]
        ucon = torch.cat([u0[..., None], ui], -1)
        ucov = (g[0] * ucon[..., None, :]).sum(-1)
        b0 = (p[..., 5:8] * ucov[..., 1:]).sum(-1)
        bi = (p[..., 5:8] + b0[..., None] * ui) / u0[..., None]
        bcon = torch.cat([b0[..., None], bi], -1)
        return ucon, ucov, bcon, (g[0] * bcon[..., None, :]).sum(-1)

    def stress(self, p, q, d):
        ucon, ucov, bcon, bcov = q
        bsq = (bcon * bcov).sum(-1)
        pg = torch.zeros_like(bsq) if self.ffde else (self.gam - 1) * p[..., 1]
        w = torch.zeros_like(bsq) if self.ffde else p[..., 0] + p[..., 1] + pg
        delta = torch.zeros(4, dtype=p.dtype, device=p.device)
        delta[d] = 1.0
        return ((w + bsq) * ucon[..., d])[..., None] * ucov + (pg + bsq / 2)[..., None] * delta - bcon[..., d:d + 1] * bcov

    def flux(self, p, q, d, pos, at=None):
        """F of direction d (0: U), times gdet; rest mass taken out of the energy."""
        u = q[0]
        f0 = p[..., 0] * u[..., d]
        T = self.stress(p, q, d)
        if not self.ffde:
            T = torch.cat([(T[..., 0] + f0)[..., None], T[..., 1:]], -1)
        B = p[..., 5:8] if d == 0 else (p[..., 5:8] * u[..., d:d + 1] - p[..., 4 + d:5 + d] * u[..., 1:]) / u[..., :1]
        return torch.cat([f0[..., None], T, B], -1) * self.geo(pos, at)[2][..., None]

    def speeds(self, p, q, d, pos, at):
        ucon, _, bcon, bcov = q
        gcon = self.geo(pos, at)[1]
        bsq = (bcon * bcov).sum(-1)
        W = p[..., 0] + self.gam * p[..., 1]
        ok = W > 0
        cs2 = torch.where(ok, self.gam * (self.gam - 1) * p[..., 1] / torch.where(ok, W, torch.ones_like(W)), torch.zeros_like(W))
        E = bsq + torch.where(ok, W, torch.zeros_like(W))
        va2 = torch.where(E > 0, bsq / torch.where(E > 0, E, torch.ones_like(E)), torch.zeros_like(E))
        c2 = torch.clamp(cs2 + va2 - cs2 * va2, 0.0, 1.0)
        a, b = ucon[..., d], ucon[..., 0]
        A = b * b - (gcon[..., 0, 0] + b * b) * c2
        Bq = 2 * (a * b - (gcon[..., 0, d] + a * b) * c2)
        C = a * a - (gcon[..., d, d] + a * a) * c2
        s = torch.sqrt(torch.clamp(Bq * Bq - 4 * A * C, min=0.0))
        v1, v2 = (Bq - s) / (2 * A), (Bq + s) / (2 * A)
        return torch.maximum(v1, v2), torch.minimum(v1, v2)

    # -- reconstruction: values at the two faces of every zone but the outer two --
    def edges(self, p, dim):
        n = p.shape[dim]
        y = [p.narrow(dim, m, n - 4) for m in range(5)]

        def minmod(a, b):
            return torch.where(a * b <= 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))

        def slope(a, b, c):
            if self.prm.lim == H.VANL:
                s = (b - a) * (c - b)
                return torch.where(s <= 0, torch.zeros_like(s), 2 * s / torch.where(s <= 0, torch.ones_like(s), c - a))
            if self.prm.lim == H.MINM:
                return minmod(b - a, c - b)
            return minmod(0.5 * (c - a), minmod(2 * (b - a), 2 * (c - b)))
        if self.prm.lim != H.PARA:
            dq = slope(y[1], y[2], y[3])
            return y[2] - 0.5 * dq, y[2] + 0.5 * dq
        d1, d2, d3 = (slope(y[m], y[m + 1], y[m + 2]) for m in range(3))
        lo = 0.5 * (y[2] + y[1]) - (d2 - d1) / 8
        hi = 0.5 * (y[3] + y[2]) - (d3 - d2) / 8
        lo = torch.minimum(torch.maximum(y[2], y[1]), torch.maximum(torch.minimum(y[2], y[1]), lo))
        hi = torch.minimum(torch.maximum(y[2], y[3]), torch.maximum(torch.minimum(y[2], y[3]), hi))
        flat = (hi - y[2]) * (y[2] - lo) <= 0
        q, e = hi - lo, 8 * (y[2] - 0.5 * (lo + hi))
        lo = torch.where(q * (q - e) < 0, 3 * y[2] - 2 * hi, lo)
        hi = torch.where(q * (q + e) < 0, 3 * y[2] - 2 * lo, hi)
        return torch.where(flat, y[2], lo), torch.where(flat, y[2], hi)

    def faces(self, p, d):
        """F at the faces i in [0,N1] (d=1; j in [-1,N2]) or j in [0,N2] (d=2;
        i in [-1,N1]), and the largest speed there."""
        n1, n2 = self.prm.n1, self.prm.n2
        dim = d - 1
        cut = p[:, 2:n2 + 4] if d == 1 else p[2:n1 + 4]
        lo, hi = self.edges(cut, dim)  # zones -1 .. N along d
        n = lo.shape[dim]
        pl, pr = hi.narrow(dim, 0, n - 1), lo.narrow(dim, 1, n - 1)
        at = (slice(3, n1 + 4), slice(2, n2 + 4)) if d == 1 else (slice(2, n1 + 4), slice(3, n2 + 4))
        pos = d - 1
        g = self.geo(pos, at)
        bn = 0.5 * (pl[..., 4 + d] + pr[..., 4 + d])[..., None]
        F, U, cmax, cmin = [], [], [], []
        for v in (pl, pr):
            v = self.limit(torch.cat([v[..., :4 + d], bn, v[..., 5 + d:]], -1), g, self.prm.gammamax)
            q = self.state(v, pos, at)
            F.append(self.flux(v, q, d, pos, at))
            U.append(self.flux(v, q, 0, pos, at))
            a, b = self.speeds(v, q, d, pos, at)
            cmax.append(a)
            cmin.append(b)
        cp = torch.clamp(torch.maximum(*cmax), min=0.0)
        cm = torch.clamp(-torch.minimum(*cmin), min=0.0)
        top = torch.maximum(cp, cm)
        lax = 0.5 * (F[0] + F[1] - top[..., None] * (U[1] - U[0]))
        if self.prm.fluxmethod == H.HLLFLUX:
            a, b = cp[..., None], cm[..., None]
            s = torch.where(a + b == 0, torch.ones_like(a), a + b)
            return torch.where(a + b == 0, lax, (a * F[0] + b * F[1] - a * b * (U[1] - U[0])) / s), top
        return lax, top

    def fix_flux(self, F1, F2):
        P = self.prm
        n1, n2 = P.n1, P.n2
        polar = (P.bc[H.X2DN] == H.POLARAXIS, P.bc[H.X2UP] == H.POLARAXIS)
        if P.bc[H.X1DN] == H.OUTFLOW:
            F1[0, :n2 + 1, 0].clamp_(max=0.0)
        if P.bc[H.X1UP] == H.OUTFLOW:
            F1[n1, :n2 + 1, 0].clamp_(min=0.0)
        keep = torch.zeros(8, dtype=F2.dtype, device=F2.device)
        keep[3] = 1.0
        if polar[0]:
            F1[:n1, 0, 6] = -F1[:n1, 1, 6]
            F2[:n1 + 1, 0] = torch.where(keep > 0, F2[:n1 + 1, 0], torch.zeros_like(keep))
        if polar[1]:
            F1[:n1, n2 + 1, 6] = -F1[:n1, n2, 6]
            F2[:n1 + 1, n2] = torch.where(keep > 0, F2[:n1 + 1, n2], torch.zeros_like(keep))
        eq = (n2 - 1) // 2
        F2[1:n1 + 1, eq] = torch.where(keep > 0, F2[1:n1 + 1, eq], torch.zeros_like(keep))

    def change(self, pb, psrc):
        """dU/dt of the interior and the Courant limits of both directions."""
        P = self.prm
        n1, n2 = P.n1, P.n2
        F1, c1 = self.faces(pb, 1)
        F2, c2 = self.faces(pb, 2)
        if P.fixupflux:
            self.fix_flux(F1, F2)
        e1 = F1[..., 6] / self.gdet[3:n1 + 4, 2:n2 + 4, 0]
        e2 = F2[..., 5] / self.gdet[2:n1 + 4, 3:n2 + 4, 1]
        emf = 0.25 * self.gdet[3:n1 + 4, 3:n2 + 4, 2] * (e1[:, 1:] + e1[:, :-1] - e2[1:] - e2[:-1])
        F1, F2 = F1[:, 1:n2 + 1].clone(), F2[1:n1 + 1].clone()
        F1[..., 5] = 0
        F1[..., 6] = 0.5 * (emf[:, :-1] + emf[:, 1:])
        F2[..., 5] = -0.5 * (emf[:-1] + emf[1:])
        F2[..., 6] = 0
        at = (slice(3, n1 + 3), slice(3, n2 + 3))
        q = self.state(psrc, 3, at)
        T = torch.stack([self.stress(psrc, q, d) for d in range(4)], -2)          # T^j_k
        conn = self.conn[at].transpose(-1, -3).transpose(-1, -2)                    # [j][k][l] of Gamma^k_{lj}
        src = (T[..., None] * conn).sum((-2, -3)) * self.gdet[at][..., 3, None]
        dU = -(F1[1:] - F1[:-1]) / P.dx1 - (F2[:, 1:] - F2[:, :-1]) / P.dx2
        dU[..., 1:5] += src
        lim = [float(torch.clamp(P.cour * dx / c, max=1e9).min()) for dx, c in ((P.dx1, c1), (P.dx2, c2))]
        return dU, lim

    # -- conserved to primitive --
    def invert_ffde(self, U, guess, at):
        gcov, gcon, gdet = self.geo(3, at)
        V = U / gdet[..., None]
        B = torch.cat([torch.zeros_like(V[..., :1]), V[..., 5:8]], -1)
        Bc = (gcov * B[..., None, :]).sum(-1)
        Bsq = (B * Bc)[..., 1:].sum(-1)
        E = torch.cat([torch.zeros_like(V[..., :1]), torch.linalg.cross(Bc[..., 1:], V[..., 2:5], dim=-1)], -1) / (Bsq * gdet)[..., None]
        Ec = (gcov * E[..., None, :]).sum(-1)
        Esq = (E * Ec)[..., 1:].sum(-1)
        g2, most = Bsq / (Bsq - Esq), self.prm.gammamax ** 2
        real = torch.where((g2 > most) | (g2 < 1), torch.sqrt(torch.clamp(Esq * Bsq, min=0) / (1 - 1 / most)), Bsq)
        drift = torch.linalg.cross(Ec[..., 1:], Bc[..., 1:], dim=-1) / (real * gdet)[..., None]
        v = (drift - gcon[..., 0, 1:]) / (-gcon[..., 0, 0])[..., None]
        w = torch.cat([torch.ones_like(v[..., :1]), v], -1)
        ut = 1 / torch.sqrt(-(gcov * w[..., :, None] * w[..., None, :]).sum((-1, -2)))
        return torch.cat([guess[..., :2], v * ut[..., None], V[..., 5:8]], -1), torch.zeros_like(gdet, dtype=torch.int64)

    def invert(self, U, guess, at):
        """The root of the two equations in W and v^2 nearest the guess."""
        if self.ffde:
            return self.invert_ffde(U, guess, at)
        gcov, gcon, gdet = self.geo(3, at)
        V = U / gdet[..., None]
        alpha = 1 / torch.sqrt(-gcon[..., 0, 0])
        D = alpha * V[..., 0]
        B = torch.cat([torch.zeros_like(V[..., :1]), alpha[..., None] * V[..., 5:8]], -1)
        Q = alpha[..., None] * torch.cat([(V[..., 1] - V[..., 0])[..., None], V[..., 2:5]], -1)
        Qc = (gcon * Q[..., None, :]).sum(-1)
        Bsq = (B * (gcov * B[..., None, :]).sum(-1)).sum(-1)
        QB = (Q * B).sum(-1)
        Qn = -alpha * Qc[..., 0]
        Qt = (Q * Qc).sum(-1) + Qn * Qn
        utsq = self.gamma(guess, (gcov,)) ** 2 - 1
        G = self.gam
        W = (D / torch.sqrt(1 + utsq) + G * guess[..., 1]) * (1 + utsq)
        for _ in range(10):
            low = W ** 3 * (W + 2 * Bsq) - QB ** 2 * (2 * W + Bsq) <= W * W * (Qt - Bsq * Bsq)
            W = torch.where(low, 10 * W, W)
        v2 = torch.clamp((W * W * Qt + QB ** 2 * (Bsq + 2 * W)) / (W * (Bsq + W)) ** 2, 0.0, 1 - 1e-12)
        for _ in range(40):
            r = torch.sqrt(1 - v2)
            pg = (G - 1) / G * (W * (1 - v2) - D * r)
            a11 = -2 * v2 * (Bsq + W) - 2 * QB ** 2 * (Bsq + W) / W ** 3
            a12 = -(Bsq + W) ** 2
            a21 = -1 - QB ** 2 / W ** 3 + (G - 1) / G * (1 - v2)
            a22 = -Bsq / 2 + (G - 1) / G * (0.5 * D / r - W)
            f1 = Qt - v2 * (Bsq + W) ** 2 + QB ** 2 * (Bsq + 2 * W) / W ** 2
            f2 = -Qn - Bsq * (1 + v2) / 2 + QB ** 2 / (2 * W * W) - W + pg
            det = a11 * a22 - a12 * a21
            W = (W - (f1 * a22 - f2 * a12) / det).abs()
            v2 = torch.clamp(v2 - (f2 * a11 - f1 * a21) / det, 0.0, 1 - 1e-12)
        v2 = (W * W * Qt + QB ** 2 * (Bsq + 2 * W)) / (W * (Bsq + W)) ** 2
        r = torch.sqrt(1 - v2)
        rho, w = D * r, W * (1 - v2)
        u = w - rho - (G - 1) * (w - rho) / G
        ncon = -alpha[..., None] * gcon[..., 0, :]
        ut = (Qc + ncon * Qn[..., None] + (QB / W)[..., None] * B)[..., 1:] / (r * (W + Bsq))[..., None]
        bad = torch.isnan(u) | (rho <= 0) | (u < 0)
        out = torch.cat([rho[..., None], u[..., None], ut, V[..., 5:8]], -1)
        lost = torch.isnan(out).any(-1)
        out = torch.where(lost[..., None], torch.cat([guess[..., :5], V[..., 5:8]], -1), out)
        return out, bad.to(torch.int64)

    # -- ghost zones and repairs --
    def bound(self, p):
        P = self.prm
        n1, n2 = P.n1, P.n2
        rows = slice(3, n2 + 3)
        if P.bc[H.X1DN] == H.PERIODIC:
            p[:3, rows], p[n1 + 3:, rows] = p[n1:n1 + 3, rows].clone(), p[3:6, rows].clone()
        else:
            for side, at, src in ((-1, slice(0, 3), 3), (1, slice(n1 + 3, n1 + 6), n1 + 2)):
                v = p[src:src + 1, rows].expand(3, -1, -1).clone()
                g = self.geo(3, (at, rows))
                alpha = 1 / torch.sqrt(-g[1][..., 0, 0])
                ga = self.gamma(v, g)
                u1 = v[..., 2] - ga * alpha * g[1][..., 0, 1]
                fix = (u1 > 0) if side < 0 else (u1 < 0)
                w = v[..., 2:5] / ga[..., None]
                w = torch.cat([(g[1][..., 0, 1] * alpha)[..., None], w[..., 1:]], -1)
                vsq = (g[0][..., 1:, 1:] * w[..., :, None] * w[..., None, :]).sum((-1, -2))
                vsq = torch.where(vsq >= 1, torch.full_like(vsq, 1 - 1 / P.gammamax ** 2), torch.clamp(vsq, min=0.0))
                w = w / torch.sqrt(1 - vsq)[..., None]
                v[..., 2:5] = torch.where(fix[..., None], w, v[..., 2:5])
                p[at, rows] = self.limit(v, g, P.gammamax)
        if P.bc[H.X2DN] == H.PERIODIC:
            p[:, :3], p[:, n2 + 3:] = p[:, n2:n2 + 3].clone(), p[:, 3:6].clone()
        else:
            p[:, :3] = p[:, 3:6].flip(1)
            p[:, n2 + 3:] = p[:, n2:n2 + 3].flip(1)
            if P.poledeath:
                for k in (3, 6):
                    p[:, :4, k] = 0
                    p[:, n2 + 2:, k] = 0
        return p

    def repair(self, p, bad):
        P = self.prm
        n1, n2 = P.n1, P.n2
        if self.ffde or not bool(bad.any()):
            return p
        f = bad.cpu().numpy()
        per1, per2 = P.bc[H.X1DN] == H.PERIODIC, P.bc[H.X2DN] == H.PERIODIC

        def good(i, j):
            j = j % n2 if per2 else (-j - 1 if j < 0 else 2 * n2 - 1 - j if j >= n2 else j)
            i = i % n1 if per1 else min(max(i, 0), n1 - 1)
            return not f[i, j]
        old = p.clone()
        for i, j in zip(*(x.tolist() for x in np.nonzero(f))):
            def ok(*d):
                return all(good(i + a, j + b) for a, b in d)

            def mean(*d):
                return sum(old[i + 3 + a, j + 3 + b, :5] for a, b in d) / len(d)
            plus, cross = ((0, 1), (0, -1), (-1, 0), (1, 0)), ((1, 1), (1, -1), (-1, 1), (-1, -1))
            for d in (plus, cross, ((0, 1), (0, -1)), ((1, 0), (-1, 0)), ((1, 1), (-1, -1)), ((1, -1), (-1, 1)),
                      ((1, 1),), ((1, 0),), ((1, -1),), ((0, -1),), ((-1, -1),), ((-1, 0),), ((-1, 1),), ((0, 1),)):
                if ok(*d):
                    new = mean(*d)
                    break
            else:
                new = 0.5 * (mean(*plus) + mean(*cross))
            at = (slice(i + 3, i + 4), slice(j + 3, j + 4))
            g = self.geo(3, at)
            most = min(float(self.gamma(old[at], g)), P.gammamax)
            v = old[at].clone()
            v[..., :5] = new
            p[at] = self.limit(v, g, most) if most > 1 else v
        return p

    def step(self, p, dt):
        P = self.prm
        n1, n2 = P.n1, P.n2
        cuf, cn, pb_, pf_ = {
            4: ([[1, 0, .5], [1, 0, .5], [1, 0, 1], [1, 0, 1]], [[1, 1 / 6, 0], [0, 1 / 3, 0], [0, 1 / 3, 0], [0, 1 / 6, 0]],
                "paba", "abap"),
            3: ([[1, 0, 1], [.75, .25, .25], [1 / 3, 2 / 3, 2 / 3]], [[0, 0, 0], [0, 0, 0], [0, 0, 1]], "pab", "abp"),
            2: ([[1, 0, .5], [1, 0, 1]], [[0, 0, 0], [0, 0, 1]], "pa", "ap")}[P.timeorder]
        at = (slice(3, n1 + 3), slice(3, n2 + 3))
        arr = {"p": p}
        pi = p[at].clone()
        Ui = self.flux(pi, self.state(pi, 3, at), 0, 3, at)
        last, new = torch.zeros_like(Ui), torch.zeros_like(Ui)
        for s in range(len(cuf)):
            dU, lim = self.change(arr[pb_[s]], arr[pb_[s]][at])
            Uf = cuf[s][0] * Ui + cuf[s][1] * last + cuf[s][2] * dt * dU
            new = new + cn[s][0] * Ui + cn[s][1] * dt * dU + cn[s][2] * Uf
            last = Uf
            v, bad = self.invert(new if s == len(cuf) - 1 else Uf, pi, at)
            if not self.ffde:
                v[..., 0] = torch.maximum(v[..., 0], torch.clamp(self.floors[at][..., 0], min=P.rhominlimit))
                v[..., 1] = torch.maximum(v[..., 1], torch.clamp(self.floors[at][..., 1], min=P.uuminlimit))
            v = self.limit(v, self.geo(3, at), P.gammamax)
            f = torch.zeros_like(p)
            f[at] = v
            f = self.bound(f)
            arr[pf_[s]] = self.bound(self.repair(f, bad))
        return arr["p"], min(P.defcon / (1 / lim[0] + 1 / lim[1]), P.safe * dt)


def _exact_steps(problem, geom, p0, lim, flux, order, steps):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    R = _Exact(*geom.tables(), _params(problem, geom, lim, flux, order), dev)
    p = R.bound(torch.as_tensor(p0, dtype=torch.float64, device=dev).clone())
    t, dt = 0.0, FIRST_DT[problem]
    for _ in range(steps):
        p, new = R.step(p, dt)
        t, dt = t + dt, new
    return p.cpu(), np.array([t, dt])


def exact(case, seed):
    do = case["do"]
    if do == "invert":
        _, zones, _, _, pr = _inversion_inputs(case, seed)
        return {"pr": pr, "flag": np.zeros(len(zones), dtype=np.int32)}
    if do == "adjoint":  # its own tests hold it against differences and forward mode
        return None
    if do == "batch":
        got = [_exact_steps("torus", geom, p0, "para", "hll", 4, case["steps"]) for geom, p0 in _torus_states(case, seed)]
        return {"p": [g[0] for g in got], "time": np.array([g[1] for g in got])}
    geom = _geometry(case["problem"], case["n1"], case["n2"], _spin(case["problem"]))
    p, time = _exact_steps(case["problem"], geom, _state(case["problem"], geom, seed), case["lim"], case["flux"],
                           case["order"], case["steps"])
    return {"p": p, "time": time}
