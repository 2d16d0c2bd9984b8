"""What programs ask of this library, as cases that can be timed and checked.

A case is one whole call sequence of a user's program on host fields, the form in which every host of the
library (the Fortran one, the Python package) holds them: the state goes up, the solve runs on the device, the
state comes back.  Handles (a solver, a batch, a server) are made once in prepare(), as such programs keep
them.  The tile of the stage kernel is the library's own choice, which is what a program driven by an input
deck gets.  exact() restates the scheme in plain torch FP64: edge reconstruction, edge flux, divergence, the
Runge-Kutta stages and the CFL time step of the compressible Euler equations on a structured grid.
"""
import math
import random

import numpy as np
import torch

from fvleg_2d_amd import SchemeConfig, Solver
from fvleg_2d_amd.batch import Batch
from fvleg_2d_amd.serve import Server

GAMMA = 1.4
PERIODIC = "periodic,periodic,periodic,periodic"  # +x, -x, +y, -y
OPEN = "zero_gradient,zero_gradient,zero_gradient,zero_gradient"
CHANNEL = "zero_gradient,zero_gradient,periodic,periodic"
WALLS = "symmetry,symmetry,zero_gradient,symmetry"

MIXED_FLUXES = ("AUSM+", "AUSMPW+", "HLLC", "Roe")
MIXED_LIMITERS = ("minmod", "MLP5")


# ---- the cases ------------------------------------------------------------------------------------------
def _solve(name, form, flow, ni, nj, flux, limiter, integrator, bcs, cfl, steps, precision="fp64", grid="uniform",
           max_time=0.0):
    return {"name": name, "form": form, "flow": flow, "ni": ni, "nj": nj, "flux": flux, "limiter": limiter,
            "integrator": integrator, "bcs": bcs, "cfl": cfl, "steps": steps, "precision": precision, "grid": grid,
            "max_time": max_time}


def listed():
    return [
        # the shock tube every newcomer runs first, to its end: 1600 cells, some 690 steps, launches and latency
        _solve("shock_tube", "loop", "tube", 400, 4, "AUSM+", "minmod", "ssp_rk2", CHANNEL, 0.4, 0, max_time=0.2),
        # a host-driven time loop (get_timestep, integrate) on a small closed box with the input deck's defaults
        _solve("host_loop", "steps", "riemann", 161, 95, "AUSMPW+", "minmod", "ssp_rk2", WALLS, 0.1, 24),
        # the small 2D problem of a parameter study: odd sizes, a multistage integrator
        _solve("small_2d", "loop", "riemann", 301, 243, "Roe", "superbee", "rk(2,4)", OPEN, 0.4, 96),
        # a four-quadrant Riemann problem, FP64 and with the edge arithmetic in FP32
        _solve("riemann", "loop", "riemann", 1024, 1024, "HLLC", "MLP5", "ssp_rk3", OPEN, 0.4, 128),
        _solve("riemann_fp32", "loop", "riemann", 1024, 1024, "HLLC", "MLP5", "ssp_rk3", OPEN, 0.4, 128, "fp32_flux"),
        # a Kelvin-Helmholtz layer at the size production runs take, in both precisions
        _solve("shear_layer", "loop", "shear", 2048, 2048, "SLAU", "van_leer", "ssp_rk3", PERIODIC, 0.5, 192),
        _solve("shear_layer_fp32", "loop", "shear", 2048, 2048, "SLAU", "van_leer", "ssp_rk3", PERIODIC, 0.5, 192,
               "fp32_flux"),
        # a ragged ordinary grid whose sides divide by nothing
        _solve("ragged", "loop", "riemann", 1237, 611, "SLAU2", "MLP3", "ssp_rk3", OPEN, 0.4, 96),
        # body-fitted cells: volumes, lengths and normals read per cell
        _solve("curvilinear", "loop", "shear", 500, 421, "SLAU", "van_leer", "ssp_rk3", PERIODIC, 0.5, 96,
               grid="wavy"),
        # one call of the flux solver from a host that keeps its own time integrator
        _solve("flux_solver", "residual", "riemann", 640, 481, "SLAU", "minmod", "ssp_rk2", WALLS, 0.4, 1),
        # a parameter study in one batch: uneven grids and mixed schemes
        {"name": "batch", "form": "batch", "count": 32, "lo": 64, "hi": 256, "mix": 2024, "steps": 64,
         "precision": "fp64"},
        # requests answered by a resident server
        {"name": "server", "form": "serve", "count": 8, "lo": 128, "hi": 384, "mix": 77, "steps": 0,
         "max_time": 0.02, "precision": "fp32_flux"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(("loop", "loop", "loop", "loop", "steps", "residual", "batch", "serve"))
    if form == "batch":
        return {"form": form, "count": rng.randint(5, 40), "lo": rng.randint(40, 90), "hi": rng.randint(120, 300),
                "mix": rng.randrange(1 << 20), "steps": rng.randint(20, 70),
                "precision": rng.choice(("fp64", "fp32_flux"))}
    if form == "serve":
        return {"form": form, "count": rng.randint(2, 9), "lo": rng.randint(100, 160), "hi": rng.randint(200, 400),
                "mix": rng.randrange(1 << 20), "steps": 0, "max_time": rng.uniform(0.008, 0.02),
                "precision": rng.choice(("fp64", "fp32_flux"))}
    # sides from a strip of a few cells to the largest grid, each on its own
    limiter = rng.choice(("minmod", "superbee", "van_leer", "MLP3", "MLP5"))
    cells = _log_int(rng, 1500, 1 << (21 if limiter.startswith("MLP") else 22))
    nj = max(4, min(2048, int(math.sqrt(cells) * math.exp(rng.uniform(-0.7, 0.7)))))
    ni = max(16, min(2048, cells // nj))
    if form == "steps":
        ni, nj = min(ni, 703), min(nj, 699)
    flow = rng.choice(("riemann", "shear", "tube"))
    grid = "wavy" if form == "loop" and flow == "shear" and ni * nj < 400000 and rng.random() < 0.4 else "uniform"
    flux = "SLAU" if grid == "wavy" else rng.choice(("AUSM+", "AUSMPW+", "HLLC", "Roe", "SLAU", "SLAU2"))
    bcs = {"shear": PERIODIC, "tube": CHANNEL}.get(flow) or rng.choice((OPEN, WALLS))
    return _solve("", form, flow, ni, nj, flux, limiter, rng.choice(("ssp_rk2", "ssp_rk3", "rk(1,3)", "rk(2,4)")),
                  bcs, round(rng.uniform(0.1, 0.5), 3), 1 if form == "residual" else rng.randint(16, 128),
                  rng.choice(("fp64", "fp64", "fp32_flux")), grid)


# ---- inputs ---------------------------------------------------------------------------------------------
def _n_ghost(limiter):
    return 3 if limiter == "MLP5" else 2


def _nodes(ni, nj, nh, grid, height):
    """Node coordinates with nh ghost layers: uniform cells over [0, 1] x [0, height], or those displaced."""
    x = np.linspace(-nh / ni, 1.0 + nh / ni, ni + 1 + 2 * nh)
    y = np.linspace(-nh * height / nj, height * (1.0 + nh / nj), nj + 1 + 2 * nh)
    x, y = np.meshgrid(x, y, indexing="ij")
    if grid == "wavy":
        s = np.sin(2 * np.pi * y / height)
        x, y = (x + 0.03 * np.sin(2 * np.pi * x) * s, y + 0.03 * height * np.sin(2 * np.pi * x + 1.0) * s)
    return np.asfortranarray(x), np.asfortranarray(y)


def _quadrants(ni, nj, rng):
    """Four states, one to a quadrant: densities in [0.3, 2], speeds in [-0.7, 0.7], pressures in [0.3, 1.5],
    so that no corner opens a vacuum."""
    state = np.column_stack((rng.uniform(0.3, 2.0, 4), rng.uniform(-0.7, 0.7, 4), rng.uniform(-0.7, 0.7, 4),
                             rng.uniform(0.3, 1.5, 4)))
    right, top = np.arange(ni) >= ni // 2, np.arange(nj) >= nj // 2
    q = np.asfortranarray((2 * right[:, None] + top[None, :]).astype(np.int8))
    return [np.asfortranarray(state[:, k][q]) for k in range(4)]


def _shear(ni, nj, rng):
    """A dense stream between two slower ones, disturbed by eight sine modes and a little noise."""
    x, y = (np.arange(ni) + 0.5) / ni, (np.arange(nj) + 0.5) / nj
    inner = np.abs(y - 0.5) < 0.25
    wave = sum(np.sin(2 * np.pi * (m + 1) * x + rng.uniform(0, 2 * np.pi)) for m in range(8))
    one = np.ones((ni, nj), order="F")
    v = np.asfortranarray(rng.random((nj, ni)).T)
    v *= 2e-3
    v += (0.01 * wave - 1e-3)[:, None]
    return [one * np.where(inner, 2.0, 1.0), one * np.where(inner, 0.5, -0.5), v, one * 2.5]


def _tube(ni, nj, rng):
    """A shock tube along x in a cross-stream that shears at the diaphragm, its left state scattered a little."""
    one = np.ones((ni, nj), order="F")
    left = ((np.arange(ni) + 0.5) / ni < 0.5)[:, None]
    rho, p = np.where(left, rng.uniform(0.9, 1.1), 0.125), np.where(left, rng.uniform(0.9, 1.1), 0.1)
    return [one * rho, one * 0.0, one * np.where(left, 0.2, -0.1), one * p]


def _problem(case, seed):
    """The config, grid and initial primitives of one solve, by name."""
    ni, nj, nh = case["ni"], case["nj"], _n_ghost(case["limiter"])
    height = nj / ni  # square cells, whatever the sides
    rng = np.random.default_rng([seed, ni, nj])
    fields = {"riemann": _quadrants, "shear": _shear, "tube": _tube}[case["flow"]](ni, nj, rng)
    x, y = _nodes(ni, nj, nh, case["grid"], height)
    return {"case": case, "x": x, "y": y, "fields": fields}


def _members(case, seed):
    """The solves of a batch or a server's queue: square sides log-uniform in [lo, hi], schemes drawn."""
    mix, out = random.Random(case["mix"]), []
    for k in range(case["count"]):
        side = _log_int(mix, case["lo"], case["hi"])
        one = _solve("", "loop", "riemann", side, side, mix.choice(MIXED_FLUXES), mix.choice(MIXED_LIMITERS),
                     "ssp_rk3", OPEN, 0.4, case["steps"], case["precision"],
                     max_time=case.get("max_time", 0.0) * mix.uniform(0.5, 1.0))
        out.append(_problem(one, seed * 1000 + k))
    return out


def _config(case):
    return SchemeConfig(flux=case["flux"], limiter=case["limiter"], integrator=case["integrator"],
                        bcs=tuple(case["bcs"].split(",")), gamma=GAMMA, cfl=case["cfl"], precision=case["precision"])


class _Request:
    """A solve as Batch and Server take it."""

    def __init__(self, pb):
        self.cfg, self.node_x, self.node_y = _config(pb["case"]), pb["x"], pb["y"]
        self.rho, self.u, self.v, self.p = pb["fields"]
        self.max_time = pb["case"]["max_time"]


# ---- one pass -------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["form"] in ("batch", "serve"):
        members = [_Request(pb) for pb in _members(case, seed)]
        if case["form"] == "batch":
            return {"case": case, "members": members, "batch": Batch(members, precision=case["precision"])}
        return {"case": case, "members": members,
                "server": Server(1e9, max_slots=16, precision=case["precision"], steps_per_tick=8)}
    pb = _problem(case, seed)
    pb["solver"] = Solver(_config(case), pb["x"], pb["y"])
    if case["form"] == "residual":
        nh = _n_ghost(case["limiter"])
        pb["halo"] = [np.asfortranarray(np.pad(f, nh)) for f in pb["fields"]]
    return pb


def _loop_limits(case):
    return (case["max_time"], 0) if case["max_time"] else (1e300, case["steps"])


def run(state):
    case = state["case"]
    if case["form"] == "batch":
        b, members = state["batch"], state["members"]
        for k, m in enumerate(members):
            b.set_primitive(k, m.rho, m.u, m.v, m.p)
        n, t, err = b.run(1e300, 1e300, max_iterations=case["steps"])
        return {"state": _joined([b.conserved(k) for k in range(len(members))]), "steps": n, "time": t, "error": err}
    if case["form"] == "serve":
        s = state["server"]
        ids = [s.submit(m) for m in state["members"]]
        s.drain()
        ends = [s.poll(i) for i in ids]
        return {"state": _joined([s.result(i) for i in ids]), "steps": np.array([e[2] for e in ends]),
                "error": np.array([e[3] for e in ends])}
    s = state["solver"]
    if case["form"] == "residual":
        halo = state["halo"]
        return {"ddt": s.residual(*halo), "filled": halo}
    s.set_primitive(*state["fields"])
    if case["form"] == "steps":
        t, err = 0.0, 0
        for _ in range(case["steps"]):
            dt = s.compute_dt()
            err |= s.step(dt)
            t += dt
        return {"state": s.conserved(), "time": t, "error": err}
    n, t, err = s.run(*_loop_limits(case))
    return {"state": s.conserved(), "steps": n, "time": t, "error": err}


def _joined(results):
    """The fields of several solves, one after another, by variable."""
    return [np.concatenate([r[k].ravel(order="F") for r in results]) for k in range(4)]


# ---- what a pass cannot do without ----------------------------------------------------------------------
# floating-point operations of one edge's flux, and of both its states for one variable, counted in exact()
FLUX_FLOPS = {"AUSM+": 90, "AUSMPW+": 120, "HLLC": 95, "Roe": 150, "SLAU": 110, "SLAU2": 110}
RECON_FLOPS = {"minmod": 17, "superbee": 23, "van_leer": 21, "MLP3": 46, "MLP5": 72}
CELL_FLOPS = 70  # divergence, stage combination, primitives
STAGES = {"ssp_rk2": 2, "ssp_rk3": 3, "rk(1,3)": 3, "rk(2,4)": 4}


def _solve_work(case, steps):
    cells, stages = case["ni"] * case["nj"], STAGES[case["integrator"]]
    flops = cells * stages * steps * (2 * (FLUX_FLOPS[case["flux"]] + 4 * RECON_FLOPS[case["limiter"]]) + CELL_FLOPS)
    # a stage reads U_0 and U_k (one state in the first) and writes U_k+1; the host's fields go up and down once
    return {"bytes": cells * (steps * (96 * stages - 32) + 64), "flops": flops}


def work(case):
    if case["form"] in ("batch", "serve"):
        total = {"bytes": 0, "flops": 0}
        for pb in _members(case, 0):
            c = pb["case"]
            w = _solve_work(c, c["steps"] or _steps_to(c))
            total = {k: total[k] + w[k] for k in total}
        return total
    if case["form"] == "residual":
        one = _solve_work(case, 1)
        return {"bytes": 64 * case["ni"] * case["nj"], "flops": one["flops"] / STAGES[case["integrator"]]}
    return _solve_work(case, case["steps"] or _steps_to(case))


def _steps_to(case):
    """Steps to max_time at waves of about |u| + c = 2 in x and, where the flow is two-dimensional, in y."""
    return max(1, int(case["max_time"] * case["ni"] * (4.0 if case["flow"] == "riemann" else 3.5) / case["cfl"]))


# ---- the same numbers in plain torch FP64 ---------------------------------------------------------------
def _pad_axis(q, ax, nh, hi, lo, flip):
    n = q.shape[ax]

    def side(kind, near):  # near: cells next to the side, outermost ghost first at the low end
        if kind == "periodic":
            return q.narrow(ax, n - nh, nh) if near == "lo" else q.narrow(ax, 0, nh)
        if kind == "zero_gradient":
            edge = q.narrow(ax, 0 if near == "lo" else n - 1, 1)
            return torch.cat([edge] * nh, ax)
        ghost = torch.flip(q.narrow(ax, 0 if near == "lo" else n - nh, nh), (ax,))
        return -ghost if flip else ghost

    return torch.cat([side(lo, "lo"), q, side(hi, "hi")], ax)


def _fill(prims, bcs, nh):
    """rho, u, v, p with nh ghost layers on every side."""
    out = []
    for k, q in enumerate(prims):
        q = _pad_axis(q, 0, nh, bcs[0], bcs[1], k == 1)
        out.append(_pad_axis(q, 1, nh, bcs[2], bcs[3], k == 2))
    return out


def _stencil(q, ax, nh):
    """at(a, b): q at normal offset a and transverse offset b from the cell left of each edge along ax."""
    n, m = q.shape[ax] - 2 * nh, q.shape[1 - ax] - 2 * nh

    def at(a, b=0):
        return q.narrow(ax, nh - 1 + a, n + 1).narrow(1 - ax, nh + b, m)

    return at


def _tvd(at, limiter):
    def phi(r):
        if limiter == "minmod":
            return r.clamp(0.0, 1.0)
        if limiter == "superbee":
            return torch.maximum((2 * r).clamp(0.0, 1.0), r.clamp(0.0, 2.0))
        return (r + r.abs()) / (1 + r.abs())

    dm, dp, d3 = at(0) - at(-1), at(1) - at(0), at(2) - at(1)
    return at(0) + 0.5 * phi(dp / (dm + 1e-16)) * dm, at(1) - 0.5 * phi(dp / (d3 + 1e-16)) * d3


def _mlp(at, order):
    tiny, eps = 1e-30, 2.0 ** -52

    def diff(a, b):  # a difference at round-off level counts as none
        d = at(a) - at(b)
        return torch.where(d.abs() < eps, torch.zeros_like(d), d)

    dm, dp, d3 = diff(0, -1), diff(1, 0), diff(2, 1)
    rr, rl = dp / (d3 + tiny), dp / (dm + tiny)
    if order == 5:
        rl_m, rr_p = dm / (diff(-1, -2) + tiny), d3 / (diff(3, 2) + tiny)
        beta_l = (-2 / (rl_m + tiny) + 11 + 24 * rl - 3 * rl * (d3 / (dp + tiny))) / 30
        beta_r = (-2 / (rr_p + tiny) + 11 + 24 * rr - 3 * rr * (dm / (dp + tiny))) / 30
    else:
        beta_l, beta_r = (1 + 2 * rl) / 3, (1 + 2 * rr) / 3
    t0 = (at(0, 1) - at(0, -1)).abs() / ((at(1) - at(-1)).abs() + tiny)
    t1 = (at(1, 1) - at(1, -1)).abs() / ((at(2) - at(0)).abs() + tiny)

    def limited(r, other, here, there, beta, d):
        a = (2 * r.clamp(min=1.0) * (1 + (there / (other + tiny)).clamp(min=0.0)) / (1 + here)).clamp(1.0, 2.0)
        return 0.5 * torch.minimum(torch.minimum(a * r, a), beta).clamp(min=0.0) * d

    return at(0) + limited(rl, rr, t0, t1, beta_l, dm), at(1) - limited(rr, rl, t1, t0, beta_r, d3)


def _edge_states(prims, ax, nh, limiter):
    make = (lambda at: _mlp(at, 5 if limiter == "MLP5" else 3)) if limiter.startswith("MLP") else (
        lambda at: _tvd(at, limiter))
    both = [make(_stencil(q, ax, nh)) for q in prims]
    return [b[0] for b in both], [b[1] for b in both]


def _slau(L, R, n, second):
    (rl, ul, vl, pl), (rr, ur, vr, pr), (nx, ny) = L, R, n
    ql, qr = ul * nx + vl * ny, ur * nx + vr * ny
    c = 0.5 * (torch.sqrt(GAMMA * pl / rl) + torch.sqrt(GAMMA * pr / rr))
    speed = torch.sqrt(0.5 * (ul * ul + vl * vl + ur * ur + vr * vr))
    chi = (1 - (speed / c).clamp(max=1.0)) ** 2
    q_bar = (rl * ql.abs() + rr * qr.abs()) / (rl + rr)
    p_bar, rho_bar, ml, mr = 0.5 * (pl + pr), 0.5 * (rl + rr), ql / c, qr / c
    bl = torch.where(ml.abs() < 1, 0.25 * (2 - ml) * (ml + 1) ** 2, (ml >= 0).double())
    br = torch.where(mr.abs() < 1, 0.25 * (2 + mr) * (mr - 1) ** 2, (mr < 0).double())
    dp = torch.where((pr - pl).abs() < 5e-3 * p_bar, torch.zeros_like(pl), pr - pl)
    if second:
        p = p_bar + 0.5 * (bl - br) * (pl - pr) + speed * (bl + br - 1) * rho_bar * c
    else:
        p = p_bar + 0.5 * (bl - br) * (pl - pr) + (1 - chi) * (bl + br - 1) * p_bar
    g = -ml.clamp(-1.0, 0.0) * mr.clamp(0.0, 1.0)
    m = 0.5 * (rl * ql + rr * qr - q_bar * (rr - rl)) * (1 - g) - chi / (2 * c) * dp
    fl, fr = 0.5 * (m + m.abs()), 0.5 * (m - m.abs())
    return fl + fr, fl * ul + fr * ur + p * nx, fl * vl + fr * vr + p * ny, fl * _enthalpy(L) + fr * _enthalpy(R)


def _enthalpy(s):
    return GAMMA / (GAMMA - 1) * s[3] / s[0] + 0.5 * (s[1] * s[1] + s[2] * s[2])


def _hllc(L, R, n):
    nx, ny = n

    def side(s):
        r, u, v, p = s
        q, E = u * nx + v * ny, p / (GAMMA - 1) + 0.5 * r * (u * u + v * v)
        return q, E, torch.sqrt(GAMMA * p / r), (r * q, r * u * q + p * nx, r * v * q + p * ny, q * (E + p))

    (ql, El, cl, FL), (qr, Er, cr, FR) = side(L), side(R)
    (rl, ul, vl, pl), (rr, ur, vr, pr) = L, R
    ps = (0.5 * (pl + pr) - 0.5 * (qr - ql) * 0.5 * (rl + rr) * 0.5 * (cl + cr)).clamp(min=0.0)

    def factor(p):
        return torch.where(ps <= p, torch.ones_like(p),
                           torch.sqrt((1 + (GAMMA + 1) / (2 * GAMMA) * (ps / p - 1)).clamp(min=1.0)))

    sl, sr = ql - cl * factor(pl), qr + cr * factor(pr)
    ml, mr = rl * (sl - ql), rr * (sr - qr)
    star = (pr - pl + ql * ml - qr * mr) / (ml - mr)

    def middle(s, q, E, m, speed, F):
        r, u, v, p = s
        a = m / (speed - star)
        U = (a, a * (u + (star - q) * nx), a * (v + (star - q) * ny), a * (E / r + (star - q) * (star + p / m)))
        return [f + speed * (us - u0) for f, us, u0 in zip(F, U, (r, r * u, r * v, E))]

    mid = [torch.where(star >= 0, a, b) for a, b in zip(middle(L, ql, El, ml, sl, FL), middle(R, qr, Er, mr, sr, FR))]
    return [torch.where(sl >= 0, a, torch.where(sr <= 0, b, m)) for a, b, m in zip(FL, FR, mid)]


def _ausm_plus(L, R, n):
    (rl, ul, vl, pl), (rr, ur, vr, pr), (nx, ny) = L, R, n
    ql, qr, Hl, Hr = ul * nx + vl * ny, ur * nx + vr * ny, _enthalpy(L), _enthalpy(R)
    al, ar = (torch.sqrt(2 * (GAMMA - 1) / (GAMMA + 1) * H.abs()) for H in (Hl, Hr))
    a = torch.minimum(al * al / torch.maximum(al, ql), ar * ar / torch.maximum(ar, -qr))
    Ml, Mr = ql / a, qr / a
    pos, neg = (lambda M: 0.25 * (M + 1) ** 2), (lambda M: -0.25 * (M - 1) ** 2)
    m = torch.where(Ml.abs() >= 1, Ml.clamp(min=0.0), pos(Ml) * (1 - 2 * neg(Ml))) + torch.where(
        Mr.abs() >= 1, Mr.clamp(max=0.0), neg(Mr) * (1 + 2 * pos(Mr)))
    m = torch.where(m.abs() < 1e-13, torch.zeros_like(m), m)
    p = pl * torch.where(Ml.abs() >= 1, (Ml > 0).double(), pos(Ml) * (2 - Ml - 3 * Ml * neg(Ml))) + pr * torch.where(
        Mr.abs() >= 1, (Mr < 0).double(), neg(Mr) * (-2 - Mr + 3 * Mr * pos(Mr)))
    up = m > 0
    f = m * a * torch.where(up, rl, rr)
    return f, f * torch.where(up, ul, ur) + nx * p, f * torch.where(up, vl, vr) + ny * p, f * torch.where(up, Hl, Hr)


def _ausmpw_plus(L, R, n, ax, near):
    (rl, ul, vl, pl), (rr, ur, vr, pr), (nx, ny) = L, R, n
    (Ul, Vl), (Ur, Vr) = ((ul, vl), (ur, vr)) if ax == 0 else ((vl, ul), (vr, ur))
    mach = [torch.sqrt(u * u + v * v) / torch.sqrt(GAMMA * p / r) for r, u, v, p in (L, R)]
    low = (mach[0] < 0.1) | (mach[1] < 0.1)  # the low-Mach fix, on by default
    f = torch.maximum(mach[0], mach[1]).clamp(max=1.0)

    def fixed(a, b, sign):
        return torch.where(low, 0.5 * (a + b) + sign * f * 0.5 * (a - b), a if sign > 0 else b)

    ul, ur, vl, vr = fixed(ul, ur, 1), fixed(ul, ur, -1), fixed(vl, vr, 1), fixed(vl, vr, -1)
    Hl, Hr = _enthalpy((rl, ul, vl, pl)), _enthalpy((rr, ur, vr, pr))
    cs = torch.sqrt(2 * (GAMMA - 1) / (GAMMA + 1) * torch.minimum(Hl - 0.5 * Vl * Vl, Hr - 0.5 * Vr * Vr))
    c = cs * cs / torch.maximum(torch.where(Ul + Ur < 0, Ur.abs(), Ul.abs()), cs)
    Ml, Mr = Ul / c, Ur / c
    bump = lambda M: 0.125 * M * (M * M - 1) ** 2  # noqa: E731
    Mp = torch.where(Ml.abs() > 1, Ml.clamp(min=0.0), 0.25 * (Ml + 1) ** 2)
    Mm = torch.where(Mr.abs() > 1, Mr.clamp(max=0.0), -0.25 * (Mr - 1) ** 2)
    Pp = torch.where(Ml.abs() > 1, (Ml > 0).double(), 0.25 * (Ml + 1) ** 2 * (2 - Ml) + bump(Ml))
    Pm = torch.where(Mr.abs() > 1, (Mr < 0).double(), 0.25 * (Mr - 1) ** 2 * (2 + Mr) - bump(Mr))
    ps = pl * Pp + pr * Pm
    w = 1 - torch.minimum(pl / pr, pr / pl) ** 3
    around = torch.minimum(torch.minimum(near(0, 1), near(0, -1)), torch.minimum(near(1, 1), near(1, -1)))
    damp = (around / torch.minimum(pl, pr)).clamp(max=1.0) ** 2
    fl, fr = (pl / ps - 1) * damp, (pr / ps - 1) * damp
    back = Mp + Mm < 0
    ml = torch.where(back, Mp * w * (1 + fl), Mp + Mm * ((1 - w) * (1 + fr) - fl)) * c * rl
    mr = torch.where(back, Mm + Mp * ((1 - w) * (1 + fl) - fr), Mm * w * (1 + fr)) * c * rr
    p = Pp * pl + Pm * pr
    return ml + mr, ml * ul + mr * ur + nx * p, ml * vl + mr * vr + ny * p, ml * Hl + mr * Hr


def _roe(L, R, n, ax, near):
    (rl, ul, vl, pl), (rr, ur, vr, pr), (nx, ny) = L, R, n
    hl, hr = _enthalpy(L), _enthalpy(R)
    rho, d = torch.sqrt(rl * rr), torch.sqrt(rl * rr) / rl
    u, v, h = ((a + d * b) / (1 + d) for a, b in ((ul, ur), (vl, vr), (hl, hr)))
    k = 0.5 * (u * u + v * v)
    c2 = (GAMMA - 1) * (h - k)
    c, q = torch.sqrt(c2), u * nx + v * ny
    dq, dt = (ur - ul) * nx + (vr - vl) * ny, -(ur - ul) * ny + (vr - vl) * nx
    cl, cr = torch.sqrt(GAMMA * pl / rl), torch.sqrt(GAMMA * pr / rr)
    e1 = torch.minimum(q - c, ul * nx + vl * ny - cl).abs()
    e4 = torch.maximum(q + c, ur * nx + vr * ny + cr).abs()
    w2 = e1 * (pr - pl - rho * c * dq) / (2 * c2)
    w3 = q.abs() * (rr - rl - (pr - pl) / c2)
    w4 = q.abs() * rho
    w5 = e4 * (pr - pl + rho * c * dq) / (2 * c2)
    damp = (w2 + w3 + w5, w2 * (u - c * nx) + w3 * u + w4 * (ur - ul - dq * nx) + w5 * (u + c * nx),
            w2 * (v - c * ny) + w3 * v + w4 * (vr - vl - dq * ny) + w5 * (v + c * ny),
            w2 * (h - c * q) + w3 * k + w4 * (u * (ur - ul) + v * (vr - vl) - q * dq) + w5 * (h + c * q))
    fl = (rl * q, rl * ul * q + nx * pl, rl * vl * q + ny * pl, rl * hl * q)
    fr = (rr * q, rr * ur * q + nx * pr, rr * vr * q + ny * pr, rr * hr * q)
    F = [0.5 * (a + b - x) for a, b, x in zip(fr, fl, damp)]
    # a shock sensor over the edge's pressures switches a shear term on

    def jump(a, b):
        return ((a - b).abs() / (torch.minimum(a, b) + 1e-16) >= 1).double()

    on = jump(near(0, 0), near(1, 0))
    for b in (1, -1):
        beyond = jump(near(0, b), near(1, b)) if ax == 0 else jump(near(1, 0), near(1, b))
        on = torch.maximum(on, torch.maximum(jump(near(0, 0), near(0, b)), beyond))
    psi = (cr - cl).abs() / torch.maximum(cr, cl)
    F[1] = F[1] - 0.5 * on * rho * c * (-dt * ny + psi * dq * nx)
    F[2] = F[2] - 0.5 * on * rho * c * (dt * nx + psi * dq * ny)
    return F


def _geometry(x, y, nh, device):
    """Per cell, ghosts too: edge lengths (bottom, right, top, left), volume, least widths; per cell the unit
    normals of its right and its top edge."""
    x, y = torch.from_numpy(x).to(device), torch.from_numpy(y).to(device)
    X = [x[:-1, :-1], x[1:, :-1], x[1:, 1:], x[:-1, 1:]]
    Y = [y[:-1, :-1], y[1:, :-1], y[1:, 1:], y[:-1, 1:]]
    vol = (X[1] - X[0]) * (Y[3] - Y[0]) - (X[3] - X[0]) * (Y[1] - Y[0])
    e = [(X[(k + 1) % 4] - X[k], Y[(k + 1) % 4] - Y[k]) for k in range(4)]
    length = [torch.sqrt(a * a + b * b) for a, b in e]
    inner = (slice(nh, -nh), slice(nh, -nh))
    normal = [[(e[k][1] / length[k]), (-e[k][0] / length[k])] for k in (1, 2)]
    edges = [[c[nh - 1:-nh, nh:-nh] for c in normal[0]], [c[nh:-nh, nh - 1:-nh] for c in normal[1]]]
    widths = (torch.minimum(e[0][0].abs(), e[2][0].abs())[inner], torch.minimum(e[3][1].abs(), e[1][1].abs())[inner])
    return {"vol": vol[inner], "len": [q[inner] for q in length], "normal": edges, "widths": widths}


def _rate(prims, geo, case):
    """d/dt of the conserved variables, and the primitives with their ghosts filled."""
    nh = _n_ghost(case["limiter"])
    q = _fill(prims, case["bcs"].split(","), nh)
    F = []
    for ax in (0, 1):
        L, R = _edge_states(q, ax, nh, case["limiter"])
        n = geo["normal"][ax] if case["grid"] != "uniform" else (1.0 - ax, float(ax))
        near = _stencil(q[3], ax, nh)
        F.append({"SLAU": lambda: _slau(L, R, n, False), "SLAU2": lambda: _slau(L, R, n, True),
                  "HLLC": lambda: _hllc(L, R, n), "AUSM+": lambda: _ausm_plus(L, R, n),
                  "AUSMPW+": lambda: _ausmpw_plus(L, R, n, ax, near), "Roe": lambda: _roe(L, R, n, ax, near)}[case["flux"]]())
    b, r, t, l = geo["len"]
    rate = [-((f[1:] * r - f[:-1] * l) + (g[:, 1:] * t - g[:, :-1] * b)) / geo["vol"] for f, g in zip(*F)]
    return rate, q


def _to_prims(U):
    u, v = U[1] / U[0], U[2] / U[0]
    return [U[0], u, v, U[0] * (GAMMA - 1) * (U[3] / U[0] - 0.5 * (u * u + v * v))]


def _stages(integrator):
    """(weight of U^n, weight of U_k, weight of the rate) of each stage."""
    if integrator == "ssp_rk2":
        return [(0, 1, 1), (0.5, 0.5, 0.5)]
    if integrator == "ssp_rk3":
        return [(0, 1, 1), (0.75, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3)]
    return [(1, 0, a) for a in {"rk(1,3)": (0.1481, 0.4, 1.0), "rk(2,4)": (0.1084, 0.2602, 0.5052, 1.0)}[integrator]]


def _exact_solve(pb):
    case = pb["case"]
    nh = _n_ghost(case["limiter"])
    dev = "cuda" if case["ni"] * case["nj"] > 20000 and torch.cuda.is_available() else "cpu"
    geo = _geometry(pb["x"], pb["y"], nh, dev)
    prims = [torch.from_numpy(np.ascontiguousarray(f)).to(dev) for f in pb["fields"]]
    if case["form"] == "residual":
        rate, filled = _rate(prims, geo, case)
        around = (nh, nh, nh, nh)
        return {"ddt": [torch.nn.functional.pad(r, around).cpu().numpy() for r in rate],
                "filled": [f.cpu().numpy() for f in filled]}
    rho, u, v, p = prims
    U = [rho, rho * u, rho * v, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)]
    end, most = _loop_limits(case)
    n, t = 0, 0.0
    while t < end and (not most or n < most):
        c = torch.sqrt(GAMMA * prims[3] / prims[0])
        rate = (prims[1].abs() + c) / geo["widths"][0] + (prims[2].abs() + c) / geo["widths"][1]
        dt = case["cfl"] / float(rate.max())
        Un = U
        for a, b, w in _stages(case["integrator"]):
            L, _ = _rate(prims, geo, case)
            U = [a * x + b * y + (w * dt) * z for x, y, z in zip(Un, U, L)]
            prims = _to_prims(U)
        n, t = n + 1, min(t + dt, end)
    out = {"state": [x.cpu().numpy() for x in U], "time": t, "error": None}
    return out if case["form"] == "steps" else {**out, "steps": None}


def exact(case, seed):
    if case["form"] in ("batch", "serve"):
        ends = [_exact_solve(pb) for pb in _members(case, seed)]
        out = {"state": _joined([e["state"] for e in ends]), "steps": None, "error": None}
        return out if case["form"] == "serve" else {**out, "time": np.array([e["time"] for e in ends])}
    return _exact_solve(_problem(case, seed))
