"""Work that users of psph have it do, through its public Python entry points.

``listed()`` names the cases, ``draw(rng)`` makes one more of the same ranges,
``prepare(case, seed)`` builds what a program holds before the call (a loaded
``psph.Solver``), ``run(state)`` makes one pass and returns the state it left,
``work(case)`` is the least such a pass has to move and compute, and
``exact(case, seed)`` gives the same outputs from plain 64-bit torch where
that is possible.

Kinds of pass:

* ``step``: ``Solver.step()`` of the 3D plume on a state resident in HBM, then
  the zero-copy view of the particle arrays, as a program does that advances
  the plume and looks at the fields on the GPU.  The inputs are a plume that
  has been erupting for a while, as a program has it after a restart: a hot
  column of mixed erupted material above the vent, turbulent velocities and
  smoothing lengths as an adaptation leaves them (about 700 kernel-box pairs
  per particle).  ``erupt`` says whether the inlet still runs, ``wall``
  whether the wall ghosts are refreshed every step.
* ``adapt``: the neighbour search and the adaptive smoothing lengths, the
  stages a plume run adds every 50 steps.
* ``sod``: a whole 1D shock-tube run from host arrays back to host arrays.
* ``adjoint``: gradients of the plume height over a few steps with
  checkpoints, from the state in HBM.
* ``growth``: a run with domain adaptation from host arrays back to host
  arrays, in which the region of real particles grows.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "plume-sph_amd"))

import psph  # noqa: E402

FORMS = {"fp64": psph.PSPH_FP64, "pair": psph.PSPH_FP32_PAIR, "exp": psph.PSPH_FP32_EXP, "pure": psph.PSPH_FP32_PURE}


def listed():
    return [
        # the shock-tube check of an installation: the smallest calls, bound by launches and latency
        {"name": "sod 900", "kind": "sod", "n_left": 800, "steps": 20},
        # a finely resolved tube, odd size
        {"name": "sod 5401", "kind": "sod", "n_left": 4801, "steps": 10},
        # the smallest plume that is of use (tests, parameter trials): mostly ghosts
        {"name": "step 1.7k fp64", "kind": "step", "n_real": 1728, "form": "fp64", "wall": False, "erupt": False},
        # a desk-side plume in the fast form, everything on
        {"name": "step 30k exp wall", "kind": "step", "n_real": 30011, "form": "exp", "wall": True, "erupt": True},
        # the fast form after the eruption has ended
        {"name": "step 77k exp", "kind": "step", "n_real": 77003, "form": "exp", "wall": False, "erupt": False},
        # the FP32-pair form, which keeps FP64 weights
        {"name": "step 150k pair wall", "kind": "step", "n_real": 150001, "form": "pair", "wall": True, "erupt": True},
        # the all-FP32 pair arithmetic
        {"name": "step 400k pure wall", "kind": "step", "n_real": 400009, "form": "pure", "wall": True, "erupt": True},
        # the parity form at the size of a production run
        {"name": "step 1M fp64 wall", "kind": "step", "n_real": 1000000, "form": "fp64", "wall": True, "erupt": True},
        # the benchmark's plume
        {"name": "step 4M exp wall", "kind": "step", "n_real": 4000000, "form": "exp", "wall": True, "erupt": True},
        # smoothing-length adaptation
        {"name": "adapt 60k fp64", "kind": "adapt", "n_real": 60013, "form": "fp64"},
        # gradients: one checkpoint interval is recomputed
        {"name": "adjoint 30k", "kind": "adjoint", "n_real": 30011, "steps": 6, "every": 3, "wall": True},
        # domain adaptation from the vent outwards
        {"name": "growth 51k", "kind": "growth", "steps": 12, "wall": True},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "step", "sod", "adapt", "adjoint"])
    if kind == "sod":
        return {"kind": kind, "n_left": _spread(rng, 400, 6400), "steps": rng.randint(5, 20)}
    if kind == "adapt":
        return {"kind": kind, "n_real": _spread(rng, 1000, 400000), "form": rng.choice(["fp64", "exp"])}
    if kind == "adjoint":
        return {"kind": kind, "n_real": _spread(rng, 1000, 60000), "steps": rng.randint(2, 6), "every": rng.randint(1, 3),
                "wall": rng.random() < 0.5}
    n_real = _spread(rng, 1000, 1000000)
    erupt = n_real >= 20000 and rng.random() < 0.7    # a coarser spacing than this does not resolve the inlet
    return {"kind": kind, "n_real": n_real, "form": rng.choice(["fp64", "exp", "exp", "pair", "pure"]),
            "wall": erupt and rng.random() < 0.7, "erupt": erupt}


# ---- inputs ------------------------------------------------------------------
def plume_config(n_real, form="fp64", wall=False, erupt=True):
    """The weak plume of the benchmark: 8 x 8 x 12 km, vent r = 54 m, 135 m/s,
    1053 K, erupted gas fraction 0.03, at the spacing that n_real asks for."""
    lx, ly, lz = 8000.0, 8000.0, 12000.0
    cfg = psph.default_config(3)
    cfg.h_air = (lx * ly * lz / n_real) ** (1.0 / 3.0)
    for k, (lo, hi) in enumerate([(-lx / 2, lx / 2), (-ly / 2, ly / 2), (0.0, lz)]):
        cfg.dom_lo[k], cfg.dom_hi[k] = lo, hi
    cfg.vent_z = 0.0
    cfg.vent_r, cfg.vent_v, cfg.vent_T, cfg.ng0, cfg.vent_p = 54.0, 135.0, 1053.0, 0.03, 101325.0
    cfg.wall_bc = int(wall)
    cfg.cfl = 0.1             # a careful step: a thousand passes are some minutes of the plume's life
    if not erupt:
        cfg.erupt_end = -1.0
    psph.finalize_config(cfg)
    cfg.precision = FORMS[form]
    return cfg


LATTICE = 20261204           # seed of the air lattice where the case's own seed goes elsewhere
_BASE = {}


def _air(cfg, n_real):
    """The air lattice, ghosts and vent column of a spacing (psph.gen_plume)."""
    if n_real not in _BASE:
        if len(_BASE) > 3:
            _BASE.clear()
        _BASE[n_real] = psph.gen_plume(cfg, psph.meteo_standard(), LATTICE, 0.0)
    return _BASE[n_real].copy()


def plume_state(cfg, n_real, seed):
    """A plume under way: 1 % lattice jitter, a hot mixed column above the vent
    (isobaric, erupted material mixed in), velocities, adapted h."""
    P = _air(cfg, n_real)
    rng = np.random.default_rng(seed)
    a = P.a
    dx = cfg.h_air
    moved = a["bc"] != psph.BC_ERUPT_GHOST
    for k in "xyz":
        a[k][moved] += dx * 0.01 * rng.uniform(-1.0, 1.0, int(moved.sum()))
    # the lattice stays on its side of the domain's faces
    real = a["bc"] == psph.BC_REAL
    x, y, z = a["x"][real], a["y"][real], a["z"][real]
    top = cfg.dom_hi[2]
    width = max(2.5 * dx, 0.08 * (cfg.dom_hi[0] - cfg.dom_lo[0]))
    core = np.exp(-(x * x + y * y) / width ** 2) * (z < 0.6 * top)
    frac = np.where(core > 0.02, 0.5 * core, 0.0)
    erupted = rng.uniform(0.0, 1.0, len(x)) < frac
    ng = cfg.ng0 * frac
    ns, na = frac - ng, 1.0 - frac
    cvm = ns * cfg.cvs + ng * cfg.cvg + na * cfg.cva
    rm = ng * cfg.rg + na * cfg.ra
    T = a["T"][real] * (1.0 + 0.5 * core) * (1.0 + 0.01 * rng.standard_normal(len(x)))
    rho = a["p"][real] / (rm * T)
    a["m"][real] *= rho / a["rho"][real]
    a["rho"][real], a["e"][real], a["T"][real], a["xi"][real] = rho, cvm * T, T, frac
    gam = 1.0 + rm / cvm
    a["gam"][real], a["cp"][real] = gam, cvm
    a["c"][real] = np.sqrt(gam * a["p"][real] / (rho * (na + ng)))
    a["phase"][real] = np.where(erupted, 2, 1)
    a["involved"][real] = np.where(frac >= cfg.msfrc_thresh, 2, a["involved"][real])
    a["h"][real] = cfg.eta * dx * (1.0 + 0.01 * rng.uniform(-1.0, 1.0, len(x)))
    swirl = 4.0 * core
    for k, smooth in (("x", -swirl * y / width), ("y", swirl * x / width), ("z", 25.0 * core)):
        a["sv" + k][real] = smooth + 0.05 * rng.standard_normal(len(x))
        a["v" + k][real] = smooth + 0.2 * rng.standard_normal(len(x))
    return P


def sod_config(n_left):
    """Sod's tube on [-0.5, 0.5] with equal-mass particles."""
    cfg = psph.default_config(1)
    cfg.dom_lo[0], cfg.dom_hi[0] = -0.5, 0.5
    cfg.h_air = 0.5 / n_left
    cfg.eta = 1.3
    cfg.t_end = cfg.t_output = 0.2
    return psph.finalize_config(cfg)


def sod_state(cfg, seed):
    rng = np.random.default_rng(seed)
    left = (1.0, rng.uniform(0.9, 1.1), 0.0)
    P = psph.gen_shock_tube(cfg, left, (0.125, 0.1, 0.0), 0.0, 40, 20, 35, True)
    real = P["bc"] == psph.BC_REAL
    P["vx"][real] += 0.01 * rng.standard_normal(int(real.sum()))
    return P


def growth_config(wall):
    cfg = psph.default_config(3)
    cfg.h_air = 100.0
    for k, (lo, hi) in enumerate([(-1600.0, 1600.0), (-1600.0, 1600.0), (0.0, 2400.0)]):
        cfg.dom_lo[k], cfg.dom_hi[k] = lo, hi
    for k, (lo, hi) in enumerate([(-400.0, 400.0), (-400.0, 400.0), (0.0, 800.0)]):
        cfg.idom_lo[k], cfg.idom_hi[k] = lo, hi
    cfg.vent_z = 0.0
    cfg.vent_r, cfg.vent_v, cfg.vent_T, cfg.ng0, cfg.vent_p = 54.0, 135.0, 1053.0, 0.03, 101325.0
    cfg.sml_update_int = 10
    psph.finalize_config(cfg)
    cfg.adapt_domain, cfg.wall_bc = 1, int(wall)
    return cfg


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case, kind=kind)
    if kind == "sod":
        cfg = sod_config(case["n_left"])
        s["P"] = sod_state(cfg, seed)
        s["S"] = psph.Solver(cfg, len(s["P"]) + 64)
        return s
    if kind == "growth":
        cfg = growth_config(case["wall"])
        s["met"] = psph.meteo_standard()
        s["P"] = psph.gen_plume(cfg, s["met"], LATTICE, 0.01)
        real = s["P"]["bc"] == psph.BC_REAL
        for k in ("vx", "vy", "vz"):
            s["P"][k][real] += 1e-3 * np.random.default_rng(seed).standard_normal(int(real.sum()))
        s["S"] = psph.Solver(cfg, 4 * len(s["P"]) + 40000)
        return s
    cfg = plume_config(case["n_real"], case.get("form", "fp64"), case.get("wall", False), case.get("erupt", kind == "adjoint"))
    P = plume_state(cfg, case["n_real"], seed)
    S = psph.Solver(cfg, len(P) + 200000)
    S.load(P, 0.0, 0)
    if case.get("wall", False):
        S.apply_bcond()
    s["S"] = S
    return s


def _view(S):
    """The zero-copy view (the keys' bits as int32, which torch can index); each
    tensor keeps its solver, whose memory it shows."""
    view = S.device_view()
    for k, t in view.items():
        view[k] = t = t.view(torch.int32) if t.dtype == torch.uint32 else t
        t.solver = S
    return view


def run(s):
    S, kind = s["S"], s["kind"]
    if kind == "step":
        o = S.step()
        return {"dt": o.dt, "state": _view(S)}
    if kind == "adapt":
        S.search_neighs_consth()
        S.adaptive_sml()
        return {"state": _view(S)}
    if kind == "sod":
        S.load(s["P"])
        S.run(s["steps"])
        return {"state": S.read().a}
    if kind == "adjoint":
        r = S.adjoint_run(s["steps"], s["every"], grads=True)
        return {k: r[k] for k in ("H", "dH_dvent_v", "dH_dvent_T", "dH_dng0", "grad_v", "grad_sv")}
    S.load(s["P"])
    S.domain_init(s["met"], LATTICE, 0.01)
    if s["wall"]:
        S.apply_bcond()
    S.run(s["steps"])
    return {"state": S.read().a}


# ---- the least a pass has to do ------------------------------------------------
STATE_BYTES = 176.0           # 19 doubles, 3 keys, 3 flags
PAIRS = 6.0 ** 3 * 1.5 ** 3   # kernel-box pairs of a particle after an adaptation


def _plume_total(n_real):
    """Particles of plume_config(n_real) with its ghosts."""
    dx = (8000.0 * 8000.0 * 12000.0 / n_real) ** (1.0 / 3.0)
    per = 1.0
    for length in (8000.0, 8000.0, 12000.0):
        per *= 8 * math.ceil((length + 24 * dx) / (8 * dx))
    return per


def work(case):
    kind = case["kind"]
    if kind == "sod":
        n = case["n_left"] * 1.25
        # per step: five h iterations over +-6 h, RHS and density over +-3 h (h = 1.3 dx)
        return {"bytes": 2 * STATE_BYTES * n, "flops": case["steps"] * n * (5 * 16 * 8.0 + 8 * 60.0 + 8 * 12.0)}
    if kind == "growth":
        n = 52000.0
        return {"bytes": 2 * STATE_BYTES * n * 1.9, "flops": case["steps"] * 0.2 * n * PAIRS * 190.0}
    n, real = _plume_total(case["n_real"]), float(case["n_real"])
    if kind == "adapt":
        # the cell order moves every field; a particle's list holds 8.5^3 1.5^3 others
        return {"bytes": 2 * STATE_BYTES * n, "flops": real * 8.5 ** 3 * 1.5 ** 3 * 20.0}
    if kind == "adjoint":
        per = real * PAIRS
        return {"bytes": 2 * STATE_BYTES * n * case["steps"], "flops": case["steps"] * per * (2 * 190.0 + 600.0)}
    # RHS 116, density and energy smoothing 40, filter 30 flops a pair
    return {"bytes": 2 * STATE_BYTES * n, "flops": real * PAIRS * 186.0}


# ---- the same outputs from plain 64-bit torch ----------------------------------
ISP = 0.564189583547756      # the kernel's 1 / sqrt(pi) to the digits the method uses
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _eos(cfg, rho, e, xi):
    na, ng = 1 - xi, cfg.ng0 * xi
    cvm = (xi - ng) * cfg.cvs + ng * cfg.cvg + na * cfg.cva
    rm = ng * cfg.rg + na * cfg.ra
    gam = 1 + rm / cvm
    p = rm * rho * e / cvm
    return p, torch.sqrt(gam * p / (rho * (na + ng))), e / cvm, gam, cvm


def _device_order(cfg, P):
    """The order the particle arrays have in HBM after a search: by cell, then
    by the Morton code of the place inside the cell, ties as they were."""
    n = len(P)
    ext = [cfg.ext_hi[k] - cfg.ext_lo[k] for k in range(3)]
    edge = max(cfg.cutoff * P["h"].max() * (1 + 1e-9), 5.0 * math.cbrt(ext[0] * ext[1] * ext[2] / n)
               if hasattr(math, "cbrt") else 5.0 * float(np.cbrt(ext[0] * ext[1] * ext[2] / n)))
    num = [max(1, math.ceil((ext[k] + 2 * edge) / edge)) for k in range(3)]
    cells = num[0] * num[1] * num[2]
    bits = 0
    while bits < 32 and (1 << bits) <= cells:
        bits += 1
    fine = min(4, (32 - bits) // 3)
    code = np.zeros(n, np.int64)
    cell = []
    for k, name in enumerate("xyz"):
        f = (P[name] - (cfg.ext_lo[k] - edge)) * (1.0 / edge)
        c = np.clip(np.floor(f), 0, num[k] - 1)
        u = np.clip(np.floor((f - c) * (1 << fine)), 0, (1 << fine) - 1).astype(np.int64)
        for b in range(fine):
            code |= ((u >> b) & 1) << (3 * b + k)
        cell.append(c.astype(np.int64))
    key = (((cell[2] * num[1] + cell[1]) * num[0] + cell[0]) << (3 * fine)) | code
    return np.argsort(key, kind="stable")


def _pairs(cfg, A, reach, same_bucket):
    """(i, j, dx) of the candidates of every real particle i: |dx| <= reach_i on
    each axis and in its list (its bucket, or 4.25 h_i within the adjacent ones)."""
    x = torch.stack([A["x"], A["y"], A["z"]])
    lo = torch.tensor([cfg.ext_lo[k] for k in range(3)], device=x.device, dtype=x.dtype)[:, None]
    bucket = torch.floor((x - lo) / cfg.bucket_edge)
    targets = torch.nonzero(A["bc"] >= 99).flatten()
    step = max(1, int(1.5e8) // x.shape[1])
    for s in range(0, len(targets), step):
        i = targets[s:s + step]
        far = (x[:, i, None] - x[:, None, :]).abs().amax(0)
        near = far <= reach[i, None]
        ii, jj = torch.nonzero(near, as_tuple=True)
        amax, i = far[ii, jj], i[ii]
        d = (bucket[:, i] - bucket[:, jj]).abs().amax(0)
        keep = ((d == 0) | ((d <= 1) & (amax <= cfg.list_factor * A["h"][i]))) & (amax <= cfg.cutoff2 * A["h"][i])
        yield i[keep], jj[keep], (x[:, i[keep]] - x[:, jj[keep]]), amax[keep]


def _step3(cfg, P):
    o = _device_order(cfg, P)
    A = {k: torch.from_numpy(P[k][o].astype(np.int64) if P[k].dtype.kind in "ui" else P[k][o]).to(DEV) for k in P.a}
    n = len(o)
    real = A["bc"] >= 99
    dt = cfg.cfl * float((A["h"] / A["c"])[real].min())
    dt = min(dt, cfg.t_output)
    h, m, rho0, xi0 = A["h"], A["m"], A["rho"], A["xi"]
    hmax = h.max()
    v, sv = torch.stack([A["vx"], A["vy"], A["vz"]]), torch.stack([A["svx"], A["svy"], A["svz"]])
    force, power = torch.zeros_like(v), torch.zeros_like(rho0)
    r1, r2, wn, wv = (torch.zeros_like(rho0) for _ in range(4))
    energy, dv = torch.zeros_like(rho0), torch.zeros_like(v)
    vol = 1.0 / rho0
    contr = ((A["bc"] >= 99) | (A["bc"] == 1)) & ((A["phase"] == 1) | (A["phase"] == 2))
    reach = cfg.cutoff * torch.maximum(0.5 * (h + hmax), h) * (1 + 1e-9)
    held = []
    for i, j, dx, amax in _pairs(cfg, A, reach, True):
        hij = 0.5 * (h[i] + h[j])
        k = (amax / hij) <= cfg.cutoff
        i1, j1, d1, h1, a1 = i[k], j[k], dx[:, k], hij[k], amax[k]
        q = (d1 * d1).sum(0)
        w = ISP ** 3 / h1 ** 3 * torch.exp(-q / h1 ** 2)
        G = -2.0 * w / h1 ** 2
        dvel = sv[:, i1] - sv[:, j1]
        vr, vv = (d1 * dvel).sum(0), (dvel * dvel).sum(0)
        c2 = A["c"][i1] + A["c"][j1]
        mu = h1 * vr / (q + cfg.ata * h1 ** 2)
        visc = torch.where(vr < 0, (cfg.beta * mu - cfg.alpha * 0.5 * c2) * mu / (0.5 * (rho0[i1] + rho0[j1])), torch.zeros_like(mu))
        visc = visc - cfg.eps_half * vv * vol[j1]
        term = m[j1] * (A["p"][j1] * vol[j1] ** 2 + A["p"][i1] * vol[i1] ** 2 + visc)
        along = (dvel * d1).abs().sum(0)
        wr = G * q
        kf = 20.0 * cfg.eps_half / cfg.prandtl * (A["cp"][i1] + A["cp"][j1]) * vv * wr / (along * h1 * c2)
        heat = m[j1] * vol[j1] * vol[i1] * (A["T"][i1] - A["T"][j1]) * kf
        heat = torch.where((along != 0) & (wr != 0), heat, torch.zeros_like(heat))
        f = term * G * d1
        for a in range(3):
            force[a].index_add_(0, i1, -f[a])
        power.index_add_(0, i1, (f * dvel).sum(0) + heat)
        ok = contr[j1]
        r1.index_add_(0, i1, torch.where(ok & (A["phase"][j1] == 1), w * m[j1], torch.zeros_like(w)))
        r2.index_add_(0, i1, torch.where(ok & (A["phase"][j1] == 2), w * m[j1], torch.zeros_like(w)))
        e_in = ok & ((cfg.e_smooth_ratio * a1 / h1) <= cfg.cutoff)
        i2, j2 = i1[e_in], j1[e_in]
        we = (ISP * cfg.e_smooth_ratio / h1[e_in]) ** 3 * torch.exp(-cfg.e_smooth_ratio ** 2 * q[e_in] / h1[e_in] ** 2) * m[j2] * vol[j2]
        f_in = ((amax / h[i]) <= cfg.cutoff) & ((A["bc"][j] >= 99) | (A["bc"][j] == 2))
        i3, j3 = i[f_in], j[f_in]
        held.append((i2, j2, we, i3, j3, torch.exp(-(dx[:, f_in] ** 2).sum(0) / h[i3] ** 2)))
    gz = -cfg.g
    vn = torch.where(real, v + dt * force, v)
    vn[2] = torch.where(real, vn[2] + dt * gz, vn[2])
    e1 = torch.where(real, A["e"] + dt * (0.5 * power + sv[2] * gz), A["e"])
    for i2, j2, we, i3, j3, wf in held:
        wn.index_add_(0, i2, we)
        energy.index_add_(0, i2, we * e1[j2])
    rho = torch.where(real, r1 + r2, rho0)
    xi = torch.where(real, r2 / (r1 + r2), xi0)
    e = torch.where(real, energy / wn, e1)
    for i2, j2, we, i3, j3, wf in held:
        wf = wf * m[j3] / rho[j3]
        wv.index_add_(0, i3, wf)
        for a in range(3):
            dv[a].index_add_(0, i3, wf * (vn[a][j3] - vn[a][i3]))
    svn = torch.where(real, vn + dv / wv, sv)
    p, c, T, gam, cp = _eos(cfg, rho, e, xi)
    out = {"rho": rho, "e": e, "m": m, "h": h, "xi": xi}
    for k, val in (("p", p), ("c", c), ("T", T), ("gam", gam), ("cp", cp)):
        out[k] = torch.where(real, val, A[k])
    for a, k in enumerate("xyz"):
        out["v" + k], out["sv" + k] = vn[a], svn[a]
        out[k] = torch.where(real, A[k] + dt * svn[a], A[k])
    return {"dt": dt, "state": {**{k: None for k in P.a}, **{k: out[k].cpu() for k in out}}}


def _adapt3(cfg, P):
    o = _device_order(cfg, P)
    A = {k: torch.from_numpy(P[k][o].astype(np.int64) if P[k].dtype.kind in "ui" else P[k][o]).to(DEV) for k in P.a}
    real = A["bc"] >= 99
    h0, h = A["h"], A["h"].clone()
    done = ~real
    contr = (A["bc"] >= 99) | (A["bc"] == 1)
    reach = torch.maximum(cfg.list_factor * h0, torch.full_like(h0, cfg.bucket_edge))
    reach = torch.minimum(reach, cfg.cutoff * cfg.c_smooth * h0 * 1.5)
    lists = []
    for i, j, dx, amax in _pairs(cfg, dict(A, h=h0), reach, True):
        k = contr[j]
        lists.append((i[k], (dx[:, k] ** 2).sum(0), amax[k], A["m"][j[k]]))
    for _ in range(cfg.num_loop):
        H = cfg.c_smooth * h
        rho = torch.zeros_like(h)
        for i, q, amax, mj in lists:
            k = (amax / H[i]) <= cfg.cutoff
            rho.index_add_(0, i[k], (ISP / H[i[k]]) ** 3 * torch.exp(-q[k] / H[i[k]] ** 2) * mj[k])
        new = cfg.eta * (A["m"] / rho) ** (1.0 / 3.0)
        close = ((new - h) / h).abs() < cfg.thresh
        h = torch.where(done, h, cfg.ratio_sml_dx * new)
        done = done | close
    out = {k: A[k].cpu() for k in ("x", "y", "z", "m", "rho", "e", "p")}
    return {"state": {**{k: None for k in P.a}, **out, "h": h.cpu()}}


def _sod(cfg, P, steps):
    A = {k: torch.from_numpy(P[k].copy()).to(DEV) for k in ("x", "vx", "rho", "e", "m", "h", "p", "c", "gam", "T", "xi")}
    bc = torch.from_numpy(P["bc"].astype(np.int64)).to(DEV)
    x, v, rho, e, m, h, p, c, xi = (A[k] for k in ("x", "vx", "rho", "e", "m", "h", "p", "c", "xi"))
    T, gam = A["T"], A["gam"]
    t = torch.nonzero(bc >= 99).flatten()
    time = 0.0
    contr = (bc >= 99) | (bc == 0) | (bc == 1)
    for _ in range(steps):
        dt = cfg.cfl * float((h / c)[t].min())
        dt = min(dt, cfg.t_end - time)
        time += dt
        dx = x[t, None] - x[None, :]
        ax = dx.abs()
        done = torch.zeros(len(t), dtype=torch.bool, device=DEV)
        ht = h[t]
        for _ in range(cfg.num_loop):
            H = cfg.c_smooth * ht
            w = ISP / H[:, None] * torch.exp(-(dx / H[:, None]) ** 2)
            rs = torch.where(((ax / H[:, None]) <= cfg.cutoff) & contr[None], w * m[None], torch.zeros_like(w)).sum(1)
            new = cfg.eta * (m[t] / rs)
            close = ((new - ht) / ht).abs() < cfg.thresh
            ht = torch.where(done, ht, cfg.ratio_sml_dx * new)
            done = done | close
        h = h.clone()
        h[t] = ht
        hij = 0.5 * (ht[:, None] + h[None, :])
        inside = ((ax / hij) <= cfg.cutoff) & (ax <= cfg.cutoff2 * ht[:, None])
        w = torch.where(inside, ISP / hij * torch.exp(-(dx / hij) ** 2), torch.zeros_like(dx))
        G = -2.0 * w / hij ** 2
        dv = v[t, None] - v[None, :]
        vr = dx * dv
        mu = hij * vr / (dx * dx + cfg.ata * hij ** 2)
        visc = (cfg.beta * mu - cfg.alpha * 0.5 * (c[t, None] + c[None, :])) * mu / (0.5 * (rho[t, None] + rho[None, :]))
        visc = torch.where(vr < 0, visc, torch.zeros_like(visc))
        f = m[None] * ((p / rho ** 2)[None] + (p / rho ** 2)[t, None] + visc) * G * dx
        density = torch.where(contr[None], w * m[None], torch.zeros_like(w)).sum(1)
        v, e, rho = v.clone(), e.clone(), rho.clone()
        power = (f * dv).sum(1)
        v[t] = v[t] - dt * f.sum(1)
        e[t] = e[t] + dt * 0.5 * power
        rho[t] = density
        xi = xi.clone()
        xi[t] = 0.0
        q = _eos(cfg, rho, e, xi)
        p, c, T, gam = (torch.where(bc >= 99, a, b) for a, b in zip(q[:4], (p, c, T, gam)))
        x = torch.where(bc >= 99, x + dt * v, x)
    out = {"x": x, "vx": v, "rho": rho, "e": e, "m": m, "h": h, "p": p, "c": c, "gam": gam, "T": T}
    return {"state": {**{k: None for k in P.a}, **{k: out[k].cpu() for k in out}}}


def exact(case, seed):
    kind = case["kind"]
    if kind == "sod":
        cfg = sod_config(case["n_left"])
        return _sod(cfg, sod_state(cfg, seed), case["steps"])
    if kind in ("step", "adapt") and not case.get("erupt", False) and not case.get("wall", False) \
            and case["n_real"] * _plume_total(case["n_real"]) < 5e10:
        cfg = plume_config(case["n_real"], case["form"], False, False)
        P = plume_state(cfg, case["n_real"], seed)
        return _step3(cfg, P) if kind == "step" else _adapt3(cfg, P)
    return None
