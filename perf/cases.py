"""The work that is measured when this framework is made faster.

A user steps projection cases: a deck of particles goes up, the time loop runs
some steps, and pressure and velocity come back (an output interval, or the end
of a served request).  The cases below are such passes through the public
entry points (``urbansph.Case`` and ``urbansph.Batch``), over the sizes,
precisions, solvers and options that the repository's own configurations,
tests and benchmark use, from a box of 4096 particles to the street canyon of
two million.

Two kinds of pass:

* from the deck: upload, neighbour search, set-up, the steps, the fields back.
  Served requests, refined cases and moving particles are used this way, and
  a pass always starts from the same state;
* running: a large case is in the middle of its time loop (searched and
  warmed up), and a pass is the next steps of that loop and the fields back.

Results of the mixed mode come back as floats, as the reference's particle
records hold them; those of the FP64 mode as doubles.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "urban-sph_a100_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import abi  # noqa: E402
import cases as decks  # noqa: E402
import urbansph  # noqa: E402

DX = 0.008                 # spacing of the canyons, m
WARM = 6                   # steps of a running case before its first pass: search, set-up, launch tuning
FIELDS = ("PRES", "UX", "UY", "UZ")


def listed():
    return [
        # the smallest call: a box of the size smoke tests use, one FP64 step; launches and latency
        dict(name="box_4k_fp64", kind="box", nf=10, mixed=False, mg=False, steps=1),
        # the reference's CPU configuration: the 32^3 box (54,872 particles), FP64, tolerance 1e-8, one step
        dict(name="box_55k_fp64", kind="box", nf=32, mixed=False, mg=False, steps=1),
        # the same box in mixed precision with the multigrid, a few steps
        dict(name="box_55k_mixed", kind="box", nf=32, mixed=True, mg=True, steps=4),
        # a short served request: a small canyon from its deck through 20 steps
        dict(name="request_20k_mixed", kind="request", target=20000, mixed=True, mg=True, steps=20),
        # a medium one
        dict(name="request_200k_mixed", kind="request", target=200000, mixed=True, mg=True, steps=20),
        # the headline: the two-million-particle street canyon in its time loop
        dict(name="canyon_2m_mixed", kind="running", target=0, mixed=True, mg=True, steps=10),
        # the reference's own precision and preconditioner on a canyon in its time loop
        dict(name="canyon_150k_fp64", kind="running", target=150000, mixed=False, mg=False, steps=4),
        # time to the first step of a large case: upload, search, lists, matrix, hierarchy, one step
        dict(name="start_1m_mixed", kind="request", target=1000000, mixed=True, mg=True, steps=1),
        # a drop-in caller's defaults (FP64, the reference's single Jacobi sweep) with every scalar equation on
        dict(name="scalars_100k_fp64", kind="scalars", target=100000, steps=5),
        # moving particles: the search, the matrix and the hierarchy at every step
        dict(name="moving_300k_mixed", kind="moving", target=300000, steps=4),
        # a refined canyon (three resolutions around its building), first steps after the refinement
        dict(name="refined_150k_mixed", kind="refined", target=150000, steps=2),
        # an ensemble of uneven canyons stepped together
        dict(name="ensemble_16_mixed", kind="ensemble", ncases=16, lo=20000, hi=120000, steps=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "request", "request", "request", "running", "running", "scalars", "moving", "refined",
                       "ensemble"])
    if kind == "box":
        mixed = rng.random() < 0.5
        return dict(kind=kind, nf=_log(rng, 9, 40), mixed=mixed, mg=mixed, steps=rng.randint(1, 4))
    if kind == "request":
        return dict(kind=kind, target=_log(rng, 10000, 500000), mixed=True, mg=rng.random() < 0.8,
                    steps=rng.randint(4, 20))
    if kind == "running":   # large enough that a state's passes stay within a few hundred steps (see _canyon)
        if rng.random() < 0.3:
            return dict(kind=kind, target=_log(rng, 100000, 250000), mixed=False, mg=rng.random() < 0.3, steps=4)
        return dict(kind=kind, target=_log(rng, 400000, 1600000), mixed=True, mg=True, steps=rng.randint(6, 10))
    if kind == "scalars":
        return dict(kind=kind, target=_log(rng, 10000, 150000), steps=rng.randint(2, 6))
    if kind == "moving":
        return dict(kind=kind, target=_log(rng, 15000, 400000), steps=rng.randint(2, 4))
    if kind == "refined":
        return dict(kind=kind, target=_log(rng, 40000, 250000), steps=rng.randint(1, 2))
    return dict(kind=kind, ncases=rng.randint(8, 16), lo=20000, hi=_log(rng, 50000, 120000), steps=rng.randint(3, 6))


# ---------------------------------------------------------------- decks ----
@functools.lru_cache(maxsize=6)
def _canyon(target):
    """A canyon deck: about ``target`` particles around one building, or
    (target 0) the 2.0 x 1.0 x 0.5 m canyon with eight buildings.  The scheme
    is stable on these for 300 steps or more, whatever dt is."""
    return decks.canyon(dx=DX) if target == 0 else decks.sized_canyon(target, u_scale=1.0, bh=0.08, dx=DX)


def _gusts(P, r):
    """The deck's log-law wind at another strength, with a few long waves on it."""
    P = P.copy()
    s = r.uniform(0.7, 1.3)
    wave = np.zeros((3, len(P)))
    for c in range(3):
        for _ in range(3):
            k = r.uniform(2.0, 12.0, 3)
            wave[c] += r.uniform(0.01, 0.04) * np.sin(k[0] * P["x"] + k[1] * P["y"] + k[2] * P["z"] + r.uniform(0, 6.28))
    u = P["ux"].astype(np.float64)
    P["ux"] = s * u * (1.0 + wave[0])
    P["uy"] = s * u * wave[1]
    P["uz"] = np.where(P["p_type"] == 1, s * u * wave[2], 0.0)
    return P


def _canyon_case(target, seed, **opts):
    P, nrm, geom = _canyon(target)
    prm = decks.canyon_params(geom, urbansph.default_params(), dt=5e-5, tol=1e-6)
    prm.update(**opts)
    return _gusts(P, np.random.RandomState(seed % (1 << 32))), nrm, geom, prm


def _precision(case):
    return dict(precision=abi.MIXED if case["mixed"] else abi.FP64,
                ppe_precond=abi.PRECOND_MULTIGRID if case["mg"] else abi.PRECOND_JACOBI)


def _box_deck(case, seed):
    return decks.box(nf=case["nf"], seed_pos=2 * seed + 1, seed_vel=2 * seed + 2)[0]


# -------------------------------------------------------------- prepare ----
def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, steps=case["steps"], dt=5e-5, mixed=case.get("mixed", True))
    if kind == "box":
        prm = decks.box_params(urbansph.default_params(), tol=1e-8)
        prm.update(**_precision(case))
        P, nrm, s["dt"] = _box_deck(case, seed), None, 1e-4
    elif kind in ("request", "running"):
        P, nrm, geom, prm = _canyon_case(case["target"], seed, **_precision(case))
    elif kind == "scalars":
        s["mixed"] = False
        P, nrm, geom, prm = _canyon_case(
            case["target"], seed, ppe_solver=abi.PPE_REF_JACOBI, turbulence_model=abi.DDF, con_solve=1, concn_solve=1,
            boussinesq_solve=1, diff_coef=1e-5, T_con=305.0, T_con_t=1.0)
        P["temp"] = 300.0 + 2.0 * np.exp(-P["z"].astype(np.float64) / 0.05)
        P["concn"] = np.exp(-((P["x"].astype(np.float64) - 0.3 * geom["L3"]) / 0.1) ** 2)
        P["k_turb"] = 0.01
    elif kind == "moving":
        P, nrm, geom, prm = _canyon_case(case["target"], seed, precision=abi.MIXED,
                                         ppe_precond=abi.PRECOND_MULTIGRID, ale_positions=1)
        P["eli"] = (P["p_type"] == 1).astype(np.float32)
    elif kind == "refined":
        P, nrm, geom, prm = _canyon_case(case["target"], seed, precision=abi.MIXED,
                                         ppe_precond=abi.PRECOND_MULTIGRID)
        c = urbansph.Case(prm, len(P) + 300000)
        c.upload(P, normals=nrm)
        c.step(0, s["dt"])
        s["levels"] = decks.apr_targets(c.field("X"), c.field("Y"), c.field("Z"), c.ifield("P_TYPE"),
                                        c.ifield("I_TYPE"), geom["buildings"], 0.05, 0.0125,
                                        most=c.ifield("MOST_BUFFER"))
        s.update(case=c, P=P, nrm=nrm)
        return s
    else:
        return _prepare_ensemble(case, seed, s)
    s.update(case=urbansph.Case(prm, len(P)), P=P, nrm=nrm)
    if kind == "running":
        s["case"].upload(P, normals=nrm)
        for k in range(WARM):
            s["case"].step(k, s["dt"])
        s["case"].sync()
        s["count"] = WARM
    return s


def _prepare_ensemble(case, seed, s):
    r = np.random.RandomState(seed % (1 << 32))
    s["cases"] = []
    n = case["ncases"]
    for k in range(n):   # sizes spread over the range, the same for every seed
        f = (k * 0.618034) % 1.0
        target = int(math.exp(math.log(case["lo"]) + f * (math.log(case["hi"]) - math.log(case["lo"]))))
        P, nrm, geom = decks.sized_canyon(target, u_scale=1.0, bh=0.05 + 0.06 * ((k * 0.754878) % 1.0), dx=DX)
        prm = decks.canyon_params(geom, urbansph.default_params(), dt=s["dt"], tol=1e-6, precision=abi.MIXED,
                                  L=decks.STABILITY_L[k % 3])
        prm.update(ppe_precond=abi.PRECOND_MULTIGRID)
        c = urbansph.Case(prm, len(P))
        c.upload(_gusts(P, r), normals=nrm)
        s["cases"].append(c)
    s["batch"] = urbansph.Batch()
    for k in range(WARM):
        s["batch"].step(s["cases"], [k] * n, [s["dt"]] * n)
    s["batch"].sync()
    s["count"] = WARM
    return s


# ------------------------------------------------------------------ run ----
def _read(c, mixed):
    out = {f: c.field(f) for f in FIELDS}
    return {f: a.astype(np.float32) for f, a in out.items()} if mixed else out


def run(s):
    dt, steps = s["dt"], s["steps"]
    if s["kind"] == "ensemble":
        n = len(s["cases"])
        for _ in range(steps):
            s["batch"].step(s["cases"], [s["count"]] * n, [dt] * n)
            s["count"] += 1
        return [_read(c, True) for c in s["cases"]]
    c = s["case"]
    if s["kind"] == "running":
        for _ in range(steps):
            c.step(s["count"], dt)
            s["count"] += 1
        return _read(c, s["mixed"])
    c.upload(s["P"], normals=s["nrm"])
    first = 0
    if s["kind"] == "refined":
        c.step(0, dt)
        c.apr_refine(s["levels"], max_passes=200)
        first = 1
    for k in range(first, first + steps):
        c.step(k, dt)
    out = _read(c, s["mixed"])
    if s["kind"] == "scalars":
        out.update(TEMP=c.field("TEMP"), CONCN=c.field("CONCN"), VIS_T=c.field("VIS_T"), K_TURB=c.field("K_TURB"))
    if s["kind"] in ("moving", "refined"):   # where the particles are now
        out.update({f: c.field(f).astype(np.float32) for f in ("X", "Y", "Z")})
    return out


# ----------------------------------------------------------------- work ----
def work(case):
    """Per step: every particle's state read and written once and every
    entry of the pressure matrix read once; the pair sums of the force,
    divergence and pressure-gradient passes.  From a deck: the particle
    records up; always: the fields back."""
    if case["kind"] == "box":
        n = (case["nf"] + 6) ** 3
    elif case["kind"] == "ensemble":
        lo, hi = math.log(case["lo"]), math.log(case["hi"])
        n = sum(int(math.exp(lo + ((k * 0.618034) % 1.0) * (hi - lo))) for k in range(case["ncases"]))
    else:
        n = case["target"] or 2134256
    if case["kind"] == "refined":
        n += 90000
    mixed = case.get("mixed", case["kind"] != "scalars")
    pairs = 92.0 * n
    per_step = n * 2 * 20 * 8.0 + pairs * (4 if mixed else 8)
    flops = pairs * (4 * 40.0 + 10 * 2.0)
    deck = 0 if case["kind"] in ("running", "ensemble") else 152.0 * n
    return dict(bytes=deck + case["steps"] * per_step + n * len(FIELDS) * 8.0, flops=case["steps"] * flops)


# ---------------------------------------------------------------- exact ----
def exact(case, seed):
    """The box in 64 bits: the reference's step written with torch on whole
    pair lists, the pressure system solved to round-off.  The canyons' whole
    steps (open boundaries, wall model, markers) have no such value here."""
    if case["kind"] != "box":
        return None
    P = _box_deck(case, seed)
    return _box_steps(P, case["steps"], 1e-4)


def _box_cells(P):
    """float32 cell grid: binning cell and query cell per axis, cell counts."""
    f = np.float32
    dcell = f(f(f(1.1) * f(2.0)) * P["h_ref"][0]) / f(2.0)
    bins, query, N = [], [], []
    for a in ("x", "y", "z"):
        v = P[a]
        mn, mx = v[:-1].min(), v[:-1].max()
        mn, mx = min(mn, v[0]), max(mx, v[0])
        n = int(f(mx - mn) / dcell) + 1
        b = np.minimum(np.floor((v - mn) / f(mx - mn) * f(n)), f(n - 1)).astype(np.int64)
        q = np.minimum(np.floor((v - mn) / dcell), f(n - 1)).astype(np.int64)
        bins.append(np.maximum(b, 0))
        query.append(np.maximum(q, 0))
        N.append(n)
    return np.stack(bins, 1), np.stack(query, 1), N


def _box_steps(P, steps, dt):
    bins, query, N = _box_cells(P)
    order = np.argsort(bins[:, 0] + N[0] * (bins[:, 1] + N[1] * bins[:, 2]), kind="stable")
    P, bins, query = P[order], bins[order], query[order]
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def t(a):
        return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to(dev)

    x = torch.stack([t(P[a]) for a in ("x", "y", "z")], 1)
    u = torch.stack([t(P[a]) for a in ("ux", "uy", "uz")], 1)
    m, rho, h, p = t(P["m"]), t(P["rho"]), float(P["h"][0]), t(P["pres"])
    fluid = torch.from_numpy(P["p_type"] == 1).to(dev)
    bins, query = torch.from_numpy(bins).to(dev), torch.from_numpy(query).to(dev)
    n = len(P)
    mu = torch.where(fluid, 1.0e-3, 1.0e-2).double()

    # the pairs of the two windows, self pairs left out (their terms vanish)
    I, J = [], []
    for a in range(0, n, 1024):
        d = x[a:a + 1024, None, :] - x[None, :, :]
        near = ((d * d).sum(2) < (4.001 * h) ** 2).nonzero()
        I.append(near[:, 0] + a)
        J.append(near[:, 1])
    I, J = torch.cat(I), torch.cat(J)
    I, J = I[I != J], J[I != J]
    d = x[I] - x[J]
    r = d.square().sum(1).sqrt()
    in_query = ((bins[J] - query[I]).abs() <= 2).all(1)
    in_bins = ((bins[J] - bins[I]).abs() <= 2).all(1)
    wide = in_query & fluid[J] & ~fluid[I]     # the wall pressure's smoothing length is 2 h
    sel = in_query & (r < 2.0 * h)
    grad = in_bins & (r < 2.0 * h) & fluid[J]

    def total(i, v):
        return torch.zeros((n,) + v.shape[1:], dtype=torch.float64, device=dev).index_add_(0, i, v)

    def w2(rr, hh):    # Wendland-2
        q = rr / (2.0 * hh)
        return (q < 1).double() * 3.342253804929802 / (2.0 * hh) ** 3 * (1 - q) ** 4 * (1 + 4 * q)

    def dw2(rr, hh):
        q = rr / (2.0 * hh)
        return (q < 1).double() * 3.342253804929802 / (2.0 * hh) ** 4 * -20 * q * (1 - q) ** 3

    def dw6(rr, hh):   # Wendland-6 shape, Wendland-2 normalisation
        q = rr / (2.0 * hh)
        return (q < 1).double() * 3.342253804929802 / (2.0 * hh) ** 4 * -22 * q * (1 - q) ** 7 * (16 * q * q + 7 * q + 1)

    # gradient correction: inverse of the moment matrix of the fluid neighbours
    gi, gj, gd, gr = I[grad], J[grad], d[grad], r[grad]
    M = total(gi, -(m[gj] * dw2(gr, h) / (rho[gj] * gr))[:, None, None] * gd[:, :, None] * gd[:, None, :])
    eye = torch.eye(3, dtype=torch.float64, device=dev)
    good = fluid & (torch.linalg.det(M).abs() > 2.2204460492503131e-16)
    C = torch.where(good[:, None, None], torch.linalg.inv(torch.where(good[:, None, None], M, eye)), eye)

    wi, wj, wr = I[wide], J[wide], r[wide]
    wk = m[wj] / rho[wj] * w2(wr, 2.0 * h)
    keep = wr < 4.0 * h
    wi, wj, wk = wi[keep], wj[keep], wk[keep]

    def wall_pressure(pp):
        f = total(wi, wk)
        s = total(wi, wk * pp[wj])
        return torch.where(fluid, pp, torch.where(f < 1e-6, torch.zeros_like(s), s / f.clamp_min(1e-300)))

    si, sj, sd, sr = I[sel], J[sel], d[sel], r[sel]
    fi = fluid[si]
    i, j, e, q = si[fi], sj[fi], sd[fi], sr[fi]       # pairs of the fluid rows
    g = (dw2(q, h) / q)[:, None] * e
    c = torch.einsum("nab,nb->na", C[i], (dw6(q, h) / q)[:, None] * e)
    A = 2.0 * m[j] / rho[j] * (e * c).sum(1) / q ** 2
    diag = total(i, A)
    own = fluid[j]
    oi, oj, oA = i[own], j[own], A[own]
    hm = 2.0 * rho[i] * rho[j] / (rho[i] + rho[j])
    bi, bj, bw = si[~fluid[si] & fluid[sj]], sj[~fluid[si] & fluid[sj]], w2(sr[~fluid[si] & fluid[sj]], h)

    for step in range(steps):
        u_wall = -total(bi, bw[:, None] * u[bj]) / (1e-10 + total(bi, bw))[:, None]
        u = torch.where(fluid[:, None], u, u_wall)
        if step == 0:
            p = wall_pressure(p)
        du = u[i] - u[j]
        visc = 4.0 * mu[i] * mu[j] / (mu[i] + mu[j]) * m[j] / (rho[i] * rho[j]) * (e * g).sum(1) / q ** 2
        f = total(i, visc[:, None] * du)
        f = f + total(i, ((u[i] * g).sum(1) * m[j] / rho[j])[:, None] * du)
        ux = (du * e).sum(1)
        phi = h * ux / (q * q + 0.01 * h * h)
        art = torch.where(ux < 0, 0.5 * m[i] * phi * (-0.05 * 30.0 + 0.05 * phi) / (rho[i] + rho[j]), torch.zeros_like(ux))
        f = f - total(i, art[:, None] * g)
        us = torch.where(fluid[:, None], u + dt * f, u)
        rhs = total(i, m[j] / rho[j] * ((us[j] - us[i]) * c).sum(1) * hm) / dt
        rhs = rhs + total(i[~own], A[~own] * p[j[~own]])
        p = torch.where(fluid, _solve(diag, oi, oj, oA, rhs, torch.where(fluid, p, torch.zeros_like(p)), fluid, total), p)
        p = wall_pressure(p)
        force = -2.0 * m[j] / (rho[i] * rho[j]) * (p[i] * rho[j] + p[j] * rho[i]) / (rho[i] + rho[j])
        u = torch.where(fluid[:, None], us + dt * total(i, force[:, None] * g), us)
        p = wall_pressure(p)
    out = dict(PRES=p, UX=u[:, 0], UY=u[:, 1], UZ=u[:, 2])
    return {k: v.cpu().numpy() for k, v in out.items()}


def _solve(diag, oi, oj, oA, rhs, x, rows, total):
    """BiCGSTAB with diagonal scaling to round-off (the system is not symmetric)."""
    diag = torch.where(rows, diag, torch.ones_like(diag))
    rhs = torch.where(rows, rhs, torch.zeros_like(rhs))

    def mul(v):
        return torch.where(rows, diag * v - total(oi, oA * v[oj]), torch.zeros_like(v))

    for _ in range(3):   # restarted: each pass starts from the true residual
        r = rhs - mul(x)
        rh, rho, alpha, om, v, s = r.clone(), 1.0, 1.0, 1.0, torch.zeros_like(r), torch.zeros_like(r)
        pk = torch.zeros_like(r)
        for _ in range(400):
            rho1 = float(rh @ r)
            if rho1 == 0.0 or float(r.norm()) <= 1e-15 * float(rhs.norm()):
                break
            pk = r + (rho1 / rho) * (alpha / om) * (pk - om * v)
            ph = pk / diag
            v = mul(ph)
            alpha = rho1 / float(rh @ v)
            s = r - alpha * v
            sh = s / diag
            t = mul(sh)
            tt = float(t @ t)
            om = float(t @ s) / tt if tt > 0.0 else 0.0
            x = x + alpha * ph + om * sh
            r = s - om * t
            rho = rho1
            if om == 0.0:
                break
    return x
