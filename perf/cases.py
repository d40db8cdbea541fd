"""The work that is timed: a disk (or a batch of disks) advanced to its next picture.

One pass is what a program built on this library does over and over: advance the state by the
steps between two pictures (``Context.run`` / ``Batch.run``, graph replay on) and fetch the
picture (``Context.store``), whose fields it then reads.  The context, with its device state
and step graph, is kept between passes; each pass continues from the state the last one left.

A case is a dict of plain values:

    precision   64 (the drop-in path) or 32 (the bulk path)
    nr, nphi, ntheta   the grid; ntheta 1 is a 2-D disk
    eos         0 locally isothermal, 3 adiabatic with the energy-consistent step (2-D)
    q, alpha    the planet's mass ratio; the viscosity parameter (0: inviscid)
    moving      the planet feels the disk (its forces are reduced from the disk each step)
    edges       radial edges: "fixed" ghost rings, "outflow", or "damped" (fixed with damping zones)
    disks       1, or the number of disks of a batch drawn as configs.c4_members draws them
    steps       steps between two pictures

FP64 disks return their fields as the picture holds them.  The FP32 path holds its fields in
FP32, so they are returned as FP32 tensors.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from penguin_2_0_amd import abi, configs

_DEFAULTS = {"precision": 64, "nr": 0, "nphi": 0, "ntheta": 1, "eos": 0, "q": 1.0e-4, "alpha": 0.0,
             "moving": False, "edges": "fixed", "disks": 1, "draw_seed": 0, "steps": 100}


def _case(name, **kw):
    return {"name": name, **_DEFAULTS, **kw}


def listed():
    return [
        # a user's first check of a build: the smallest disk of the tests, a handful of steps;
        # launches and the host path are all there is
        _case("fp64_48x144_10", nr=48, nphi=144, steps=10),
        # a coarse viscous disk with a picture every 100 steps, as a parameter study starts
        _case("fp32_visc_128x384_100", precision=32, nr=128, nphi=384, alpha=1.0e-3, steps=100),
        # the 256 x 768 disk and its 100 steps on the drop-in path
        _case("fp64_256x768_100", nr=256, nphi=768, steps=100),
        # odd sizes: one cell past a radial window, a ring that is no multiple of anything
        _case("fp64_visc_117x353_100", nr=117, nphi=353, alpha=3.0e-3, steps=100),
        # a migrating planet in a disk with damping zones: the CFL pass and the disk's forces
        # run beside the sweeps each step
        _case("fp32_moving_damped_389x1201_100", precision=32, nr=389, nphi=1201, moving=True, edges="damped",
              steps=100),
        # the benchmark's disk on the drop-in path
        _case("fp64_1024x3072_100", nr=1024, nphi=3072, steps=100),
        # the benchmark's disk on the bulk path, two pictures in its 1000 steps
        _case("fp32_1024x3072_500", precision=32, nr=1024, nphi=3072, steps=500),
        # the adiabatic disk on both paths: a small one with open edges on the drop-in path, and the
        # largest grid here on the bulk path
        _case("fp64_adiabatic_192x576_50", nr=192, nphi=576, eos=3, edges="outflow", steps=50),
        _case("fp32_adiabatic_1536x4608_200", precision=32, nr=1536, nphi=4608, eos=3, q=2.0e-4, steps=200),
        # spherical disks: the 3-D workload's shape at sizes that keep a picture near 100 MB
        _case("fp64_3d_96x288x32_10", nr=96, nphi=288, ntheta=32, q=3.0e-5, steps=10),
        _case("fp32_3d_128x384x32_50", precision=32, nr=128, nphi=384, ntheta=32, q=3.0e-5, steps=50),
        # the parameter sweep: uneven viscous disks advanced as one batch
        _case("fp32_batch_12_disks_100", precision=32, disks=12, draw_seed=4, steps=100),
    ]


def _log_between(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: any of the kinds above, at any size of their ranges."""
    kind = rng.choice(("disk64", "disk64", "disk32", "disk32", "adiabatic", "sphere", "batch"))
    q = float("%.3g" % _log_between(rng, 1.0e-5, 3.0e-4))
    alpha = rng.choice((0.0, float("%.3g" % _log_between(rng, 1.0e-4, 1.0e-2))))
    c = {**_DEFAULTS, "q": q, "alpha": alpha}
    if kind == "batch":
        c.update(precision=32, disks=rng.randint(2, 10), draw_seed=rng.randint(5, 10**6), steps=rng.randint(20, 100))
        c.update(q=0.0, alpha=0.0)   # the members draw their own
        return c
    if kind == "sphere":
        precision = rng.choice((64, 32))
        nr = int(_log_between(rng, 24, 112))
        c.update(precision=precision, nr=nr, nphi=int(nr * rng.uniform(2.0, 3.0)), ntheta=rng.randint(8, 32),
                 q=min(q, 1.0e-4), steps=rng.randint(4, 10) if precision == 64 else rng.randint(10, 50))
        return c
    precision = {"disk64": 64, "disk32": 32}.get(kind) or rng.choice((64, 32))
    nr = int(_log_between(rng, 40, 1000))
    nphi = int(nr * rng.uniform(2.0, 3.0))
    most = 50 * 1024 * 3072 if precision == 64 else 100 * 1024 * 3072   # zone-updates of a pass
    steps = int(_log_between(rng, 10, 200))
    c.update(precision=precision, nr=nr, nphi=nphi, steps=max(10, min(steps, most // (nr * nphi))),
             eos=3 if kind == "adiabatic" else 0)
    if kind != "adiabatic":
        c.update(moving=rng.random() < 0.2, edges=rng.choice(("fixed", "fixed", "outflow", "damped")))
    return c


def _members(case):
    """(grid, parameters) of every disk of the case."""
    if case["disks"] > 1:
        ws = configs.c4_members(seed=case["draw_seed"], n=case["disks"])
        return [(w.grid, w.params) for w in ws]
    nr, nphi, ntheta = case["nr"], case["nphi"], case["ntheta"]
    over = {"visc_flag": 1, "ss_alpha": case["alpha"], "vis_nu": case["alpha"] * 0.05 * 0.05} if case["alpha"] > 0 else {}
    if case["moving"]:
        over["plnt_flag"] = 2
    if case["edges"] == "outflow":
        over.update(nlft=1, nrgh=1)
    elif case["edges"] == "damped":
        over["kill_flag"] = 1
    if ntheta > 1:
        p = configs.c3().params.replace(M_p=case["q"], **over)
    elif case["eos"] == 3:
        p = configs.c5e3().params.replace(M_p=case["q"], **over)
    else:
        p = configs.disk2d(nr, nphi, q=case["q"], **over)
    return [(abi.PnGrid(nr, nphi, ntheta), p)]


def prepare(case, seed):
    """The disk's initial state (seeded noise of 1e-4 on Sigma) in a context, ready to run."""
    members = _members(case)
    disks = [abi.init_disk(g, p, seed * 1000 + n, 1.0e-4) for n, (g, p) in enumerate(members)]
    if case["disks"] > 1:
        batch = abi.Batch([g for g, _ in members], [p for _, p in members])
        for c, d in zip(batch.disks, disks):
            c.load(d)
        return {"steps": case["steps"], "batch": batch, "run": batch.run_begin(), "fields": "ruv"}
    (grid, params), = members
    ctx = abi.Context(grid, params, abi.PN_FP64 if case["precision"] == 64 else abi.PN_FP32)
    ctx.load(disks[0])
    fields = "ruv" + ("w" if case["ntheta"] > 1 else "p" if case["eos"] == 3 else "")
    return {"steps": case["steps"], "ctx": ctx, "run": ctx.run_begin(), "fields": fields}


def _fp32_picture(rings, fields):
    out = {f: torch.from_numpy(rings[f]).to(torch.float32) for f in fields}
    out["rot_j"] = rings["rot_j"]
    return out


def run(state):
    """Advance to the next picture and fetch it."""
    if "batch" in state:
        b, st = state["batch"], state["run"]
        b.run(state["steps"], st)
        return {"disks": [_fp32_picture(c.store(), state["fields"]) for c in b.disks],
                "time": torch.tensor([s.simtime for s in st], dtype=torch.float32)}
    ctx, st = state["ctx"], state["run"]
    ctx.run(state["steps"], st)
    rings = ctx.store()
    if ctx.precision == abi.PN_FP32:
        return {**_fp32_picture(rings, state["fields"]), "time": torch.tensor(st.simtime, dtype=torch.float32)}
    return {**{f: rings[f] for f in state["fields"]}, "rot_j": rings["rot_j"], "time": st.simtime}


def work(case):
    """Bytes: every sweep of every step reads and writes each carried field of each cell once,
    and the picture is written once (72 bytes a cell).  Flops: a sweep updates a cell with six
    parabolae, the interface solve, the Lagrangian step and the remap, about 600 operations."""
    word = case["precision"] // 8
    cells = sum(g.imax * g.jmax * g.kmax for g, _ in _members(case))
    three = case["ntheta"] > 1
    sweeps = 3 if three else 2
    fields = 3 + (1 if three or case["eos"] == 3 else 0)
    return {"bytes": cells * (case["steps"] * sweeps * 2 * fields * word + 72), "flops": cells * case["steps"] * sweeps * 600.0}


# ---------------------------------------------------------------------------------------
# The same pass in plain numpy, 64 bits: the 2-D disk with a planet fixed in the co-rotating
# frame and fixed ghost rings (the published PPMLR method, Colella & Woodward 1984, in the
# 128-cell windows of the code this library replaces).  Arrays of a window are (pencil, cell).

_NPAD, _WIN = 6, 128


def _prev(x):
    return np.concatenate((x[:, :1], x[:, :-1]), axis=1)


def _next(x):
    return np.concatenate((x[:, 1:], x[:, -1:]), axis=1)


def _within(n, lo, hi):
    c = np.arange(n)
    return (c >= lo) & (c < hi)


def _paraset(dx):
    """The interpolation coefficients of CW84 eqs. 1.6-1.7 on cells of width dx."""
    xp, an = _next(dx), dx + _next(dx)
    bn, cn = an + dx, an + xp
    anm, anp = _prev(an), _next(an)
    d = 1.0 / (anm + anp)
    c0 = dx / an * (1.0 + 2.0 * d * xp * (anm / bn - anp / cn))
    e = dx / (anm + xp)
    return c0, -d * dx * anm / bn, d * xp * anp / cn, e * _prev(bn) / an, e * cn / anm


def _parabola(lo, hi, flat, a, P):
    """Left value, jump and curvature of each cell's parabola, valid on [lo + 2, hi - 2)."""
    n = a.shape[1]
    in_coef, in_lim = _within(n, lo + 1, hi - 2), _within(n, lo + 1, hi - 1)
    dr, dl = _next(a) - a, a - _prev(a)
    s = np.where(in_lim, P[3] * dr + P[4] * dl, 0.0)
    s = np.sign(s) * np.minimum(np.abs(s), np.minimum(2.0 * np.abs(dl), 2.0 * np.abs(dr)))
    s = np.where(dl * dr < 0.0, 0.0, s)
    ar = a + np.where(in_coef, P[0] * dr + P[1] * _next(s) + P[2] * s, 0.0)
    al = flat * a + (1.0 - flat) * _prev(ar)
    ar = flat * a + (1.0 - flat) * ar
    t2, t1 = (ar - al) ** 2, (ar - al) * (6.0 * (a - 0.5 * (ar + al)))
    peak = (ar - a) * (a - al) <= 0.0
    ar, al = np.where(peak, a, ar), np.where(peak, a, al)
    al = np.where(t2 < t1, 3.0 * a - 2.0 * ar, al)
    ar = np.where(t2 < -t1, 3.0 * a - 2.0 * al, ar)
    ok = _within(n, lo + 2, hi - 2)
    return np.where(ok, al, 0.0), np.where(ok, ar - al, 0.0), np.where(ok, 6.0 * (a - 0.5 * (ar + al)), 0.0)


def _derivatives(x, u):
    """First and second derivative of the quadratic through cells c-1, c, c+1."""
    x2, x3 = x - _prev(x), _next(x) - _prev(x)
    h2, h3 = (u - _prev(u)) / x2, (_next(u) - _prev(u)) / x3
    A = (h3 - h2) / (x3 - x2)
    return 2.0 * A * x2 + (x3 * h2 - x2 * h3) / (x3 - x2), 2.0 * A


def _riemann(P, pl, rl, ul, pr, rr, ur):
    if P.eos == 0:   # two isothermal rarefactions
        t1 = 0.5 * (np.sqrt(pl / rl) + np.sqrt(pr / rr))
        t2 = -0.5 * (ur - ul) / t1
        pm = np.sqrt(pl * pr) * np.exp(t2)
        return pm, ul - t1 * np.log(pm / pl)
    g, gm = P.gam, P.gam - 1.0
    z = gm / (2.0 * g)
    cl, cr = np.sqrt(g * pl / rl), np.sqrt(g * pr / rr)
    pm = ((cl + cr - 0.5 * gm * (ur - ul)) / (cl * pl ** -z + cr * pr ** -z)) ** (1.0 / z)

    def wave(p, r, c):
        return np.where(pm > p, (pm - p) * np.sqrt(2.0 / (r * ((g + 1.0) * pm + gm * p))),
                        2.0 * c * ((pm / p) ** z - 1.0) / gm)

    return pm, 0.5 * (ur + ul) + 0.5 * (wave(pr, rr, cr) - wave(pl, rl, cl))


def _window(P, axis, W, dt, FrRot, planet):
    """One window's update in place.  W: r, p, u (along the sweep), v, w and the geometry."""
    r, p, u = W["r"], W["p"], W["u"]
    n = r.shape[1]
    x0, dx0, dvol0, rad, azi, vrot = (W[k] for k in ("x", "dx", "dvol", "rad", "azi", "vrot"))
    m, px, py, rs2 = planet

    def force(radius, angle, l):
        cosd = np.cos(angle - py)
        R3 = (radius ** 2 + px * px - 2.0 * px * radius * cosd + rs2) ** 1.5
        if axis == 0:
            return -m * (radius - px * cosd) / R3 - m * cosd / px ** 2 - 1.0 / radius ** 2 + l * l / radius ** 3
        sind = np.sin(angle - py)
        return -m * px * sind / R3 + m * sind / px ** 2

    flat = np.zeros_like(r)
    if P.flat_flag:
        dp1, dp2 = _next(p) - _prev(p), _next(_next(p)) - _prev(_prev(p))
        dp2 = np.where(np.abs(dp2) < 1.0e-15, 1.0e-15, dp2)
        shock = (np.abs(dp1) / np.minimum(_next(p), _prev(p)) > 0.33) & ~(_prev(u) < _next(u))
        steep = np.where(shock & _within(n, 2, n - 2), np.maximum(0.0, (dp1 / dp2 - 0.75) * 5.0), 0.0)
        flat = np.minimum(0.5, np.maximum(np.maximum(_prev(steep), steep), _next(steep)))
        flat = np.where(_within(n, 2, n - 2), flat, 0.0)
    # the interface states: traced averages of the parabolae and half a step of the force
    P0 = _paraset(dx0)
    if axis == 0:
        f = force(x0, azi + 0.5 * dt * vrot, 0.5 * (W["v"] + _prev(W["v"])))
    else:
        f = force(rad, x0 + 0.5 * dt * vrot, 0.0)
    cs = 0.5 * dt * np.sqrt(P.gam * p / r) / dx0
    if axis == 1:
        cs = cs / rad
    fac = 1.0 - 4.0 / 3.0 * cs

    def states(a):
        al, da, a6 = _parabola(0, n, flat, a, P0)
        return _prev(al + da - cs * (da - fac * a6)), al + cs * (da + fac * a6)

    pl, pr = (np.maximum(1.0e-15, s) for s in states(p))
    rl, rr = (np.maximum(1.0e-15, s) for s in states(r))
    ul, ur = (s + 0.5 * dt * f for s in states(u))
    pm, um = _riemann(P, pl, rl, ul, pr, rr, ur)
    pm = np.maximum(1.0e-15, pm)
    # the Lagrangian step
    move = dt * um if axis == 0 else dt * (um / rad - vrot - FrRot)
    edge = np.where(_within(n, 3, n - 2), x0 + move, x0 + 0.5 * dx0)
    inner = _within(n, 3, n - 3)
    dxl = np.where(inner, _next(edge) - edge, dx0)
    xl = np.where(inner, edge, x0)
    xc = xl + 0.5 * dxl
    if axis == 0:
        f1, f2 = force(rad, azi, W["v"]), force(xc, azi + dt * vrot, W["v"])
        dvol, area = dxl * (xl + 0.5 * dxl), 0.5 * (xl + x0)
    else:
        f1, f2 = force(rad, azi, 0.0), force(rad, xc + dt * vrot, 0.0)
        dvol, area = dxl * rad, np.ones_like(xl)
    dtdm = dt / (r * dvol0)
    un = u + 0.5 * dt * (f1 + f2) - dtdm * (_next(pm) - pm) * 0.5 * (_next(area) + area)
    q = None
    if P.eos == 3:
        e = p / (r * (P.gam - 1.0)) + 0.5 * u * u
        e = e - dtdm * (_next(area * um * pm) - area * um * pm) + 0.5 * dt * (u * f1 + un * f2)
        q = np.maximum((P.gam - 1.0) * (e - 0.5 * un * un), 1.0e-15)
    r = np.where(inner, np.maximum(r * (dvol0 / dvol), 1.0e-15), r)
    u = np.where(inner, un, u)
    # the remap to the Eulerian grid
    P1 = _paraset(dxl)
    d = xl - x0
    lvol = d * (x0 + 0.5 * d) if axis == 0 else d * rad
    ahead = d >= 0.0
    s = 0.5 * d / np.where(ahead, _prev(dxl), dxl)
    fac = np.where(ahead, 1.0 - 4.0 / 3.0 * s, 1.0 + 4.0 / 3.0 * s)

    def face(a):
        al, da, a6 = _parabola(3, n - 3, flat, a, P1)
        return np.where(ahead, _prev(al) + _prev(da) - s * (_prev(da) - fac * _prev(a6)), al - s * (da + fac * a6))

    kept = _within(n, 6, n - 6)
    flux = face(r) * lvol
    mass = r * dvol
    rn = np.maximum(1.0e-15, (mass + flux - _next(flux)) / dvol0)
    r = np.where(kept, rn, r)

    def carry(a):
        F = face(a) * flux
        return np.where(kept, (a * mass + (F - _next(F))) / (rn * dvol0), a)

    W["r"], W["u"], W["v"] = r, carry(u), carry(W["v"])
    if q is not None:
        W["p"] = np.where(kept, np.maximum(1.0e-15, r * carry(q)), p)
    if P.visc_flag:
        nu, R = W["nu"], W["R"]
        N, rho = nu * r, r
        x = x0 if axis == 0 else x0 * R
        dn = _derivatives(x, N)[0]
        u1, u2 = _derivatives(x, W["u"])
        if axis == 0:
            om = W["v"] / R ** 2
            o1, o2 = _derivatives(x, om)
            du = 2.0 * N * u2 + 2.0 * dn * u1 + 2.0 * N * u1 / R - 2.0 * N * W["u"] / R ** 2
            dv = R * (R * N * o2 + R * dn * o1 + 3.0 * N * o1)
        else:
            v1, v2 = _derivatives(x, W["v"])
            du, dv = 2.0 * N * u2 + 2.0 * dn * u1, N * v2 + dn * v1
        W["u"] = np.where(kept, W["u"] + dt * du / rho, W["u"])
        W["v"] = np.where(kept, W["v"] + dt * dv / rho, W["v"])


def _sweep(P, axis, W, dt, FrRot, planet):
    """The window update along whole pencils (cells 6 .. n - 6 of each row are the interior)."""
    n = W["r"].shape[1] - 2 * _NPAD
    out = {k: W[k][:, _NPAD:-_NPAD].copy() for k in "rpuv"}
    real = _WIN - 2 * _NPAD
    for lo in range(0, n, real):
        k = min(real, n - lo)
        part = {key: np.ascontiguousarray(a[:, lo:lo + k + 2 * _NPAD]) for key, a in W.items()}
        _window(P, axis, part, dt, FrRot, planet)
        for key in "rpuv":
            out[key][:, lo:lo + k] = part[key][:, _NPAD:_NPAD + k]
    return out


def _noise(seed, n):
    z = (np.uint64(seed) ^ np.arange(n, dtype=np.uint64)) + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return ((z ^ (z >> np.uint64(31))) >> np.uint64(11)).astype(np.float64) * 2.0 ** -52 - 1.0


def _power(r, n):
    # libm's pow: the disk's pressure slope is a difference over 1e-8 of r, which enlarges the
    # last bits of the values it is taken from
    return np.array([math.pow(x, n) for x in r])


def _exact_disk(P, nr, nphi, seed, steps):
    f = (math.log(P.xmax) - math.log(P.xmin)) / nr
    xa = np.array([P.xmin] + [P.xmin * math.exp(f * i) for i in range(1, nr)] + [P.xmax])
    dx = np.diff(xa)
    x = np.concatenate((xa[0] - dx[0] * np.arange(6, 0, -1), xa[:-1], xa[-2] + dx[-1] * np.arange(1, 7)))
    dx = np.concatenate((np.full(6, dx[0]), dx, np.full(6, dx[-1])))
    rc = x + 0.5 * dx
    dphi = (P.ymax - P.ymin) / nphi
    y = P.ymin + np.arange(nphi) * dphi
    yc = y + 0.5 * dphi
    cs2 = P.sc_h * P.sc_h * _power(rc, -P.p_beta)

    def pressure(r):
        return P.sc_h * P.sc_h * _power(r, -P.p_beta) * _power(r, -P.p_alpha)

    rho = _power(rc, -P.p_alpha)
    slope = (pressure(rc + 1.27245e-8) - pressure(rc - 1.27245e-8)) / 2.5449e-8
    vphi = np.sqrt(1.0 / rc + rc * slope / rho)
    nu = P.vis_nu * _power(rc, P.p_alpha)
    vr = -1.5 * nu / rc if P.visc_flag else np.zeros_like(rc)
    ring = slice(_NPAD, nr + _NPAD)
    S = {k: np.repeat(a[:, None], nphi, axis=1) for k, a in (("r", rho), ("p", cs2 * rho), ("u", vr), ("v", vphi))}
    S["r"][ring] *= 1.0 + 1.0e-4 * _noise(seed, nr * nphi).reshape(nr, nphi)
    S["p"] = cs2[:, None] * S["r"]
    h = math.sqrt(P.sc_h ** 2 * P.R_p ** -P.p_beta * P.R_p ** 3)
    planet = (P.M_p, P.R_p, math.pi, (P.rs_fac * h) ** 2)
    FrRot = P.R_p ** -1.5
    rot_v, res_v = vphi - FrRot * rc, np.zeros_like(rc)
    rot_j = np.zeros(len(rc), dtype=np.int32)
    dt, time = P.endtime, 0.0
    fixed = {k: S[k].copy() for k in S}
    one = np.ones((1, nr + 12))
    for _ in range(steps):
        I = {k: S[k][ring] for k in S}
        c = np.sqrt(P.gam * I["p"] / I["r"])
        R = rc[ring][:, None]
        a = (np.abs(I["u"]) + c) / dx[ring][:, None]
        b = (np.abs(I["v"] - rot_v[ring][:, None] - FrRot * R) + c) / (dphi * R)
        dt = min(1.1 * dt, P.courant / max(a.max(), b.max()))
        width = rc * dphi / dt
        jp = rot_v / width
        inc = np.where(jp >= 0.0, np.trunc(jp + 0.5), np.trunc(jp - 0.5)).astype(np.int64)
        res_v[ring] = (np.floor(jp + 0.5) * width)[ring]
        # radial sweep: pencils are lab columns
        cols = np.ones((nphi, 1))
        W = {"r": S["r"].T, "p": S["p"].T, "u": S["u"].T, "v": (S["v"] * rc[:, None]).T, "x": cols * x, "dx": cols * dx,
             "dvol": cols * (dx * (x + 0.5 * dx)), "rad": cols * rc, "azi": yc[:, None] * one, "vrot": cols * (res_v / rc),
             "nu": cols * nu, "R": cols * rc}
        g = _sweep(P, 0, W, dt, FrRot, planet)
        for k in "ruv":
            S[k][ring] = g[k].T
        S["v"][ring] /= rc[ring][:, None]
        S["p"][ring] = S["r"][ring] * cs2[ring][:, None] if P.eos == 0 else g["p"].T
        # azimuthal sweep: pencils are rings, in the lab frame, closed on themselves
        at = np.arange(-_NPAD, nphi + _NPAD)
        turn = 2.0 * math.pi * (at // nphi)
        rows = np.ones((nr, 1))
        lab = {k: S[k][ring][:, at % nphi] for k in S}
        rr = rc[ring][:, None] * np.ones((1, len(at)))
        W = {"r": lab["r"], "p": lab["p"], "u": lab["v"], "v": lab["u"], "x": rows * (y[at % nphi] + turn),
             "azi": rows * (yc[at % nphi] + turn), "dx": np.full_like(rr, dphi), "dvol": dphi * rr, "rad": rr,
             "vrot": (res_v / rc)[ring][:, None] * np.ones_like(rr), "nu": nu[ring][:, None] * np.ones_like(rr), "R": rr}
        g = _sweep(P, 1, W, dt, FrRot, planet)
        S["r"][ring], S["v"][ring], S["u"][ring] = g["r"], g["u"], g["v"]
        S["p"][ring] = S["r"][ring] * cs2[ring][:, None] if P.eos == 0 else g["p"]
        # the integer roll
        for i in range(_NPAD, nr + _NPAD):
            for k in S:
                S[k][i] = np.roll(S[k][i], inc[i])
        rot_j[ring] = (rot_j[ring] + inc[ring]) % nphi
        rot_v[ring] = (vphi - FrRot * rc)[ring]
        time += dt
        for k in S:
            S[k][:_NPAD], S[k][-_NPAD:] = fixed[k][:_NPAD], fixed[k][-_NPAD:]
    # back to the columns the picture stores them in
    out = {k: np.stack([np.roll(S[k][i], -rot_j[i]) for i in range(_NPAD, nr + _NPAD)]) for k in S}
    return out, rot_j[ring], time


def exact(case, seed):
    """The pass in 64 bits: 2-D disks with a fixed planet and fixed edges whose steps numpy takes
    in about 15 seconds (a cell's step costs it about 2 microseconds)."""
    seconds = case["steps"] * (0.03 + 2.0e-6 * case["nr"] * case["nphi"])
    if case["disks"] > 1 or case["ntheta"] > 1 or case["moving"] or case["edges"] != "fixed" or seconds > 15.0:
        return None
    (grid, params), = _members(case)
    fields = "ruv" + ("p" if case["eos"] == 3 else "")
    with np.errstate(all="ignore"):   # cells past a window's valid range are never kept
        out, rot_j, time = _exact_disk(params, grid.imax, grid.jmax, seed * 1000, case["steps"])
    return {**{f: out[f] for f in fields}, "rot_j": rot_j, "time": time}
