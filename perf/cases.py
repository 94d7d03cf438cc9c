"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values.  Its "kind" says which public entry points a
pass goes through:

* "eval"    one force evaluation of a resident cloud (tree build, h solve,
            neighbour lists, hydro, gravity) and the results fetched, as a
            program with its own integrator does.
* "run"     a whole short simulation: load initial conditions, the setup
            evaluation with guessed h, ``count`` sph_integrate steps on the
            device, the final state fetched.
* "serve"   a batch of requests on resident clouds: admit the clouds as one
            forest, step selections of them (FP64 guard steps among mixed
            ones), fetch the states.
* "forest"  an ensemble of independent clouds evaluated together: one build
            and the restock evaluations that follow it, replayed as graphs.
* "dropin"  SEREN's own drivers on SEREN-shaped host arrays, where every
            call takes its data from the host and brings its results back.

Clouds are the repository's seeded synthetic ones (uniform, r^-2 and Plummer
spheres with turbulent velocities).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from seren_amd import engine as sx
from seren_amd import ics

CS = 0.2

EVAL = dict(kind="eval", profile="uniform", multipole="octupole", mac="gadget2",
            precision="fp64", sph="gradh", thermal="isothermal", neighbours=False)
RUN = dict(kind="run", profile="r2", multipole="octupole", mac="gadget2", precision="fp64",
           integrator="lfkdk", nlevels=1, count=48)
SERVE = dict(kind="serve", multipole="octupole", mac="gadget2", precision="mixed", nmin=2048)
FOREST = dict(kind="forest", multipole="octupole", mac="gadget2", precision="mixed", nmin=4096)


def listed():
    return [
        # the smallest clouds a server keeps and the test-sized evaluation, with
        # the neighbour lists brought back: latency and launches
        dict(EVAL, name="eval uniform 2048 fp64", n=2048, multipole="quadrupole",
             mac="geometric", neighbours=True),
        # a concentrated small cloud with sparse outskirts, whose outermost
        # particles take the long road of the h solve; odd size
        dict(EVAL, name="eval plummer 2053 fp64", n=2053, profile="plummer"),
        # an ordinary small cloud in the serving precision
        dict(EVAL, name="eval r2 16384 mixed", n=16384, profile="r2", precision="mixed"),
        # standard SPH with the energy equation (h from the neighbour number)
        dict(EVAL, name="eval standard energy 30011", n=30011, multipole="quadrupole",
             mac="geometric", sph="standard", thermal="energy"),
        # a mid-sized cloud, FP64, not a multiple of anything
        dict(EVAL, name="eval uniform 131071 fp64", n=131071),
        # a larger concentrated cloud, FP64
        dict(EVAL, name="eval plummer 300007 fp64", n=300007, profile="plummer"),
        # the largest: the benchmark's cloud in mixed precision
        dict(EVAL, name="eval r2 1048576 mixed", n=1048576, profile="r2", precision="mixed"),
        # a collapsing core followed for 60 leapfrog steps, FP64
        dict(RUN, name="run r2 4096 kdk fp64", n=4096, count=120),
        # the reference's default integrator with block time steps, mixed
        dict(RUN, name="run uniform 65536 rk mixed", n=65536, profile="uniform",
             integrator="rk", nlevels=5, count=32, precision="mixed"),
        # requests on small resident clouds
        dict(SERVE, name="serve 12 clouds", clouds=12, nmax=16384, epochs=12),
        # an ensemble of independent clouds between two tree builds
        dict(FOREST, name="forest 32 clouds mixed", clouds=32, nmax=65536, restocks=3),
        # the reference's own drivers on its own arrays
        dict(kind="dropin", name="dropin uniform 12007", n=12007, profile="uniform",
             multipole="quadrupole", mac="geometric"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval", "eval", "run", "serve", "forest", "dropin"])
    if kind == "eval":
        prec = rng.choice(["fp64", "mixed"])
        std = rng.random() < 0.2
        top = 60000 if std else (300000 if prec == "fp64" else 1000000)
        multipole, mac = rng.choice([("quadrupole", "geometric"), ("octupole", "gadget2"),
                                     ("octupole", "gadget2")])
        return dict(EVAL, n=_logint(rng, 2048, top), precision=prec, multipole=multipole, mac=mac,
                    profile=rng.choice(["uniform", "r2", "plummer"]),
                    sph="standard" if std else "gradh",
                    thermal=rng.choice(["isothermal", "isothermal", "energy"]))
    if kind == "run":
        if rng.random() < 0.5:
            return dict(RUN, n=_logint(rng, 2048, 6000), count=2 * rng.randint(16, 56),
                        precision=rng.choice(["fp64", "mixed"]))
        return dict(RUN, n=_logint(rng, 4096, 65536), profile="uniform", integrator="rk",
                    nlevels=rng.randint(1, 6), count=rng.randint(8, 32),
                    precision=rng.choice(["fp64", "mixed"]))
    if kind == "serve":
        return dict(SERVE, clouds=rng.randint(4, 12), nmax=_logint(rng, 4096, 16384),
                    epochs=rng.randint(4, 12))
    if kind == "forest":
        return dict(FOREST, clouds=rng.randint(8, 32), nmin=_logint(rng, 2500, 6000),
                    nmax=_logint(rng, 16000, 65536), precision=rng.choice(["fp64", "mixed"]),
                    restocks=rng.randint(1, 4))
    return dict(kind="dropin", n=_logint(rng, 2048, 20000),
                profile=rng.choice(["uniform", "r2", "plummer"]), multipole="quadrupole",
                mac="geometric")


# ---- inputs ----------------------------------------------------------------
def _near_h(pos, profile, n):
    """A snapshot's h: 1.2 (m / rho)^(1/3) of the profile's own density."""
    r = np.linalg.norm(pos, axis=1)
    if profile == "uniform":
        rho = np.full(n, 3.0 / (4.0 * np.pi))
    elif profile == "r2":
        rho = 1.0 / (4.0 * np.pi * np.maximum(r, 30.0 / n) ** 2)
    else:
        rho = 3.0 / (4.0 * np.pi * 1e-3) * (1.0 + (r / 0.1) ** 2) ** -2.5
    return 1.2 * (1.0 / (n * rho)) ** (1.0 / 3.0)


def _near_a(pos, profile):
    """|a| of a previous evaluation, M(<r) / r^2 of the profile."""
    r = np.linalg.norm(pos, axis=1)
    if profile == "uniform":
        return np.maximum(r, 1e-3)
    if profile == "r2":
        return 1.0 / np.maximum(r, 1e-6)
    return np.maximum(r, 1e-3) / (r * r + 0.01) ** 1.5


def _cloud(n, profile, seed, mach=2.0):
    return ics.make_cloud(n, profile, seed=seed, mach=mach, cs=CS, ngrid=32)


def _energy(n, seed):
    return 0.1 * (1.0 + 0.1 * np.random.default_rng(seed).random(n))


def _forest_sizes(case):
    rng = np.random.default_rng(1000 + case["clouds"])
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [int(round(math.exp(v))) for v in rng.uniform(lo, hi, case["clouds"])]


def _engine(case, **more):
    keys = ("multipole", "mac", "precision", "sph", "thermal")
    kw = {k: case[k] for k in keys if k in case}
    return sx.ForceEngine(abserror=1e-4, thetamaxsqd=0.25, sound_speed=CS, **kw, **more)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "eval":
        n = case["n"]
        pos, vel, mass, _ = _cloud(n, case["profile"], seed)
        eng = _engine(case)
        eng.load(pos, vel, mass, _near_h(pos, case["profile"], n))
        eng.set_agravmag(_near_a(pos, case["profile"]))
        if case["thermal"] == "energy":
            eng.set_energy(_energy(n, seed))
        st["engine"] = eng
    elif kind == "run":
        st["cloud"] = _cloud(case["n"], case["profile"], seed)
        st["engine"] = _engine(case)
        st["engine"].load(*st["cloud"])
    elif kind in ("serve", "forest"):
        profiles = ("uniform", "plummer") if kind == "serve" else ("uniform",)
        st["clouds"] = [_cloud(n, profiles[k % len(profiles)], 100 * seed + k)
                        for k, n in enumerate(_forest_sizes(case))]
        st["engine"] = _engine(case, serial=kind == "serve")   # one stream, as the server runs
        st["engine"].load_forest(st["clouds"])
        if kind == "forest":
            st["engine"].force_eval(hguess=True)
    else:
        n = case["n"]
        pos, vel, mass, _ = _cloud(n, case["profile"], seed)
        st["engine"] = _engine(case)
        st["host"] = (pos, vel, mass, _near_h(pos, case["profile"], n))
    return st


# ---- one pass --------------------------------------------------------------
def run(st):
    case, eng = st["case"], st["engine"]
    kind = case["kind"]
    if kind == "eval":
        eng.force_eval()
        out = eng.fetch(neighbours=case["neighbours"])
        if case["thermal"] == "energy":
            out["u"], out["dudt"] = eng.fetch_energy()
        return out
    if kind == "run":
        eng.load(*st["cloud"])
        eng.force_eval(hguess=True)
        eng.step_begin(case["integrator"], nlevels=case["nlevels"], nbuildstep=8)
        eng.step(case["count"])
        return eng.fetch(neighbours=False)
    if kind == "serve":
        nk = case["clouds"]
        eng.load_forest(st["clouds"])
        eng.force_eval(hguess=True)
        eng.serve_begin()
        for e in range(case["epochs"]):
            sel = [(k + e) % 3 != 0 for k in range(nk)]
            if e % 4 == 3:
                eng.set_precision("fp64")
            eng.serve_step(sel)
            if e % 4 == 3:
                eng.set_precision("mixed")
        out = eng.fetch(neighbours=False)
        out["dt"], out["time"] = eng.serve_info(nk)
        return out
    if kind == "forest":
        eng.force_eval()
        for _ in range(case["restocks"]):
            eng.force_eval(restock=True, graph=True)
        return eng.fetch(neighbours=False)
    pos, vel, mass, h = st["host"]
    state = sx.SerenState(pos, vel, mass, h, eng.pp_limit)
    sx.tree_update(eng, state)
    sx.sph_update(eng, state)
    sx.update_thermal_properties_isothermal(state, CS)
    sx.sph_hydro_forces(eng, state)
    sx.sph_grav_forces(eng, state)
    names = ("parray", "v", "a", "gpot", "agravmag", "rho", "omega", "press", "sound", "div_v",
             "drhodt", "pptot", "pplist", "porig")
    return {k: getattr(state, k) for k in names}


# ---- work a pass cannot do without ----------------------------------------
def _eval_work(n, octupole=True):
    """Inputs (position, velocity, mass, h, |a|) read and results written
    once; the pair and cell terms of one evaluation, with interaction counts
    of the size the walk counters give (cells grow with log n)."""
    cells = (260.0 if octupole else 60.0) * max(1.0, math.log2(n / 64.0))
    flops = n * (cells * (190.0 if octupole else 69.0) + 150.0 * 38.0 + 57.0 * (2 * 19.0 + 30.0)
                 + 80.0 * 70.0)
    return 8.0 * n * (9 + 24), flops


def work(case):
    kind = case["kind"]
    if kind in ("eval", "dropin"):
        b, f = _eval_work(case["n"], case["multipole"] != "quadrupole")
        return {"bytes": b, "flops": f}
    if kind == "run":
        evals = case["count"] / 2.0 if case["integrator"] == "lfkdk" else 0.7 * case["count"]
        b, f = _eval_work(case["n"])
        return {"bytes": b * (1 + evals), "flops": f * (1 + evals)}
    total = sum(_forest_sizes(case))
    mean = total / case["clouds"]
    times = 1.0 + (case["epochs"] * 2.0 / 3.0 if kind == "serve" else case["restocks"])
    b, f = _eval_work(mean)
    return {"bytes": case["clouds"] * b * times, "flops": case["clouds"] * f * times}


# ---- the same in plain 64 bits ---------------------------------------------
EXACT_MAX = 33000    # particles: all pairs in about 20 s


def _tables(dev):
    """The M4 kernel's tables (entry i at s = (2 i + 1) / 10000)."""
    s = (2.0 * torch.arange(10001, dtype=torch.float64, device=dev) + 1.0) / 10000.0
    t, near = 2.0 - s, torch.arange(10001, device=dev) < 5000
    p = 0.318309886
    pick = lambda a, b: torch.where(near, a, b)  # noqa: E731
    return dict(
        w0=p * pick(1 - 1.5 * s**2 + 0.75 * s**3, 0.25 * t**3),
        w1=p * pick(-3 * s + 2.25 * s**2, -0.75 * t**2),
        w5=pick(4 / 3 * s - 1.2 * s**3 + 0.5 * s**4,
                8 / 3 * s - 3 * s**2 + 1.2 * s**3 - s**4 / 6 - 1 / (15 * s**2)),
        w6=pick(1.4 - 2 / 3 * s**2 + 0.3 * s**4 - 0.1 * s**5,
                -1 / (15 * s) + 1.6 - 4 / 3 * s**2 + s**3 - 0.3 * s**4 + s**5 / 30),
        wh=p * pick(-3 + 7.5 * s**2 - 4.5 * s**3, -6 + 12 * s - 7.5 * s**2 + 1.5 * s**3),
        wg=pick(1.4 - 2 * s**2 + 1.5 * s**4 - 0.6 * s**5,
                1.6 - 4 * s**2 + 4 * s**3 - 1.5 * s**4 + 0.2 * s**5))


def _tree_order(pos):
    """Particles in the order of an octree's leaves (at most 8 particles, the
    root divided), each leaf's in input order."""
    n = len(pos)
    lo, hi = pos.min(0), pos.max(0)
    c = np.tile(0.5 * (lo + hi), (n, 1))
    size = 0.5 * float((hi - lo).max())
    keys = np.zeros((2, n), np.int64)
    for level in range(1, 31):
        size *= 0.5
        up = pos > c
        digit = up[:, 0] + 2 * up[:, 1] + 4 * up[:, 2]
        c += np.where(up, size, -size)
        k = 0 if level <= 21 else 1
        keys[k] = keys[k] * 8 + digit
    order = np.lexsort((keys[1], keys[0]))
    a, b = keys[0][order], keys[1][order]
    leaf = np.full(n, -1)
    for level in range(1, 31):
        ka = a >> (3 * (21 - min(level, 21)))
        new = np.r_[True, ka[1:] != ka[:-1]]
        if level > 21:
            kb = b >> (3 * (30 - level))
            new[1:] |= kb[1:] != kb[:-1]
        start = np.flatnonzero(new)
        size_of = np.diff(np.r_[start, n])
        run_of = np.cumsum(new) - 1
        done = (size_of[run_of] <= 8) & (leaf < 0)
        leaf[done] = start[run_of[done]]
    return order[np.lexsort((order, leaf))]


def _offsets(x, lo, hi):
    d = x[None, :, :] - x[lo:hi, None, :]
    return d, (d * d).sum(-1)


def _index(dr, inv_h):
    return (5000.0 * dr * inv_h).to(torch.int64).clamp_(max=10000)


def _chunks(n):
    step = max(1, (1 << 25) // n)
    return [(k, min(n, k + step)) for k in range(0, n, step)]


def _density(x, m, h, T):
    """rho(h) by the sum over all pairs inside 2 h."""
    rho = torch.zeros_like(h)
    for lo, hi in _chunks(len(h)):
        _, d2 = _offsets(x, lo, hi)
        hp = h[lo:hi, None]
        w = T["w0"][_index(d2.sqrt() + 1e-20, 1.0 / hp)]
        rho[lo:hi] = (m[None] * torch.where(d2 < 4 * hp * hp, w, 0.0)).sum(1) / h[lo:hi]**3
    return rho


def _solve_h(x, m, h, T):
    """The grad-h iteration: 20 fixed-point steps, then 20 of bisection."""
    extent = float((x.max(0).values - x.min(0).values).max())
    low, high = torch.zeros_like(h), torch.full_like(h, extent)
    todo = torch.ones_like(h, dtype=torch.bool)
    rho = torch.zeros_like(h)
    for it in range(41):
        idx = torch.nonzero(todo)[:, 0]
        if not len(idx):
            break
        r = torch.zeros(len(idx), dtype=h.dtype, device=h.device)
        step = max(1, (1 << 25) // len(h))
        for k in range(0, len(idx), step):
            p = idx[k:k + step]
            d2 = ((x[None] - x[p, None])**2).sum(-1)
            hp = h[p, None]
            w = T["w0"][_index(d2.sqrt() + 1e-20, 1.0 / hp)]
            r[k:k + step] = (m[None] * torch.where(d2 < 4 * hp * hp, w, 0.0)).sum(1) / h[p]**3
        rho[idx] = r
        hp = h[idx]
        new = 1.2 * (m[idx] / r)**0.333333333
        stop = ((hp - new).abs() / hp < 0.02) & torch.tensor(it >= 1, device=h.device)
        stop |= torch.tensor(it >= 40, device=h.device)
        if it == 20:
            new = torch.full_like(new, 0.5 * extent)
        elif it > 20:
            up = hp**3 - 1.2**3 * m[idx] / r > 0
            high[idx] = torch.where(up & ~stop, hp, high[idx])
            low[idx] = torch.where(~up & ~stop, hp, low[idx])
            new = 0.5 * (low[idx] + high[idx])
        h[idx] = torch.where(stop, hp, new)
        todo[idx] = ~stop
    return 1.2 * (m / rho)**0.333333333


def exact(case, seed):
    if case["kind"] not in ("eval", "dropin") or case["n"] > EXACT_MAX:
        return None
    n = case["n"]
    std = case.get("sph") == "standard"
    energy = case.get("thermal") == "energy"
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = _tables(dev)
    pos, vel, mass, _ = _cloud(n, case["profile"], seed)
    order = _tree_order(pos)
    put = lambda a: torch.from_numpy(np.ascontiguousarray(a[order])).to(dev)  # noqa: E731
    x, v, m = put(pos), put(vel), put(mass)
    h = put(_near_h(pos, case["profile"], n))
    gather = int(4.0 * math.pi / 3.0 * 2.4**3)   # neighbours: a sphere of 2.4 mean spacings
    zero = torch.zeros_like(h)
    if std:
        for lo, hi in _chunks(n):
            d2 = _offsets(x, lo, hi)[1]
            h[lo:hi] = 0.5 * d2.kthvalue(gather + 1, dim=1).values.sqrt()
    else:
        h = _solve_h(x, m, h, T)
    rho, som, sz, sdiv = zero.clone(), zero.clone(), zero.clone(), zero.clone()
    for lo, hi in _chunks(n):
        d, d2 = _offsets(x, lo, hi)
        hp = h[lo:hi, None]
        dr = d2.sqrt() + 1e-20
        i = _index(dr, 1.0 / hp)
        near = (dr < 2 * hp) if std else (d2 <= 4 * hp * hp)
        dvdr = ((v[None] - v[lo:hi, None]) * d).sum(-1)
        mm = torch.where(near, m[None], 0.0)
        h1 = h[lo:hi]
        rho[lo:hi] = (mm * T["w0"][i]).sum(1) / h1**3
        som[lo:hi] = (mm * T["wh"][i]).sum(1) / h1**4
        sz[lo:hi] = (mm * T["wg"][i]).sum(1) / h1**2
        sdiv[lo:hi] = -(mm * dvdr * T["w1"][i] / dr).sum(1) / h1**4
    div = sdiv / rho
    omega = torch.ones_like(h) if std else 1 + h * som / (3 * rho)
    zeta = zero if std else -(h * sz) / (3 * rho * omega)
    if energy:
        u = put(_energy(n, seed))
        press = 0.4 * rho * u
        sound = (press / rho).sqrt()
    else:
        press, sound = CS * CS * rho, torch.full_like(h, CS)
    acc, pot, count = torch.zeros_like(x), zero.clone(), torch.zeros_like(h, dtype=torch.int64)
    grav, dudt = torch.zeros_like(x), zero.clone()
    pf = press / rho**2 if std else press / rho**2 / omega
    for lo, hi in _chunks(n):
        d, d2 = _offsets(x, lo, hi)
        other = torch.ones_like(d2, dtype=torch.bool)
        other[torch.arange(hi - lo, device=dev), torch.arange(lo, hi, device=dev)] = False
        dr = d2.sqrt() + 1e-20
        dr = torch.where(other, dr, 1.0)
        hp, hj = h[lo:hi, None], h[None]
        ip, ij = dr < 2 * hp, dr < 2 * hj
        count[lo:hi] = (other & ((d2 <= 4 * hp * hp) | (d2 <= 4 * hj * hj))).sum(1)
        kp, kj = _index(dr, 1 / hp), _index(dr, 1 / hj)
        # gravity, kernel-softened inside either range
        z_p, z_j = zeta[lo:hi, None], zeta[None]
        w4p, w4j = T["w1"][kp], T["w1"][kj]
        gp = torch.where(1 / dr > 0.5 / hp, (T["w5"][kp] + z_p * w4p / hp**2) / hp**2, 1 / dr**2)
        gj = torch.where(ij, (T["w5"][kj] + z_j * w4j / hj**2) / hj**2, 1 / dr**2)
        f = torch.where(other, 0.5 * m[None] / dr * (gp + gj), 0.0)
        grav[lo:hi] = (f[..., None] * d).sum(1)
        pp = torch.where(1 / dr > 0.5 / hp, T["w6"][kp] / hp, 1 / dr)
        pj = torch.where(ij, T["w6"][kj] / hj, 1 / dr)
        pot[lo:hi] = torch.where(other, 0.5 * m[None] * (pp + pj), 0.0).sum(1)
        # hydro pair forces with artificial viscosity (alpha 1, beta 2)
        wp = torch.where(ip & other, w4p / hp**4, 0.0)
        wj = torch.where(ij & other, w4j / hj**4, 0.0)
        wm = 0.5 * (wp + wj)
        unit = d / dr[..., None]
        dvdr = ((v[None] - v[lo:hi, None]) * d).sum(-1)
        if std:
            term = m[None] * wm * (pf[lo:hi, None] + pf[None])
        else:
            term = m[None] * (pf[lo:hi, None] * wp + pf[None] * wj)
        hs = hp + hj
        base = d2 if std else dr * dr
        mu = 0.5 * hs * dvdr / (base + 0.0025 * hs * hs)
        c = 0.5 * (sound[lo:hi, None] + sound[None])
        visc = (-c * mu + 2 * mu * mu) / (0.5 * (rho[lo:hi, None] + rho[None]))
        visc = torch.where(dvdr < 0, m[None] * visc * wm, 0.0)
        acc[lo:hi] = ((term + visc)[..., None] * unit).sum(1)
        dudt[lo:hi] = (0.5 * ((term if std else 0.0) + visc) * dvdr / dr).sum(1)
    if not std:
        dudt = dudt - press * div / omega / rho
    back = lambda t: t.cpu().numpy()  # noqa: E731
    agm = grav.norm(dim=1)
    drhodt = -rho * div if std else -rho * div / omega
    if case["kind"] == "dropin":
        parray = torch.cat([x, m[:, None], h[:, None], zeta[:, None]], 1)
        return {"parray": back(parray), "v": back(v), "a": back(acc + grav), "gpot": back(pot),
                "agravmag": None, "rho": back(rho), "omega": back(omega),
                "press": back(press), "sound": back(sound), "div_v": back(div),
                "drhodt": back(drhodt), "pptot": back(count).astype(np.int32), "pplist": None,
                "porig": (order + 1).astype(np.int32)}
    out = {"porig": (order + 1).astype(np.int32), "pos": back(x), "v": back(v), "m": back(m),
           "h": back(h), "zeta": back(zeta), "rho": back(rho), "omega": back(omega),
           "div_v": back(div), "drhodt": back(drhodt), "press": back(press),
           "sound": back(sound), "a": back(acc + grav), "gpot": back(pot),
           "agravmag": back(agm) if case["mac"] != "geometric" else None,
           "pptot": back(count).astype(np.int32)}
    if case["neighbours"]:
        out["pplist"] = None
    if energy:
        out["u"], out["dudt"] = back(u), back(dudt)
    return out
