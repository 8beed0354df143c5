"""The pair passes' groups, visits and queues at their edges, against the oracle.

The passes take targets in groups of 8 and chunks of 32 of a cell, visit tiles
of 64 particles and evaluate 8 queued particles at a time; list membership and
in_support are tested per pair only where a kernel box can reach past them.
Each case moves one of these: few and odd target counts (partial groups and
chunks), list boxes and support boxes inside the kernel box, smoothing lengths
that differ from particle to particle, the options that change what a pair
adds.  Bar: neighbour sets and pair counts through the fields, every
floating-point field within the parity bar of the FP64 form (1e-10 relative);
the FP32 forms within 1e-5 relative L1, the form's bar.
"""
import sys

import numpy as np
import pytest

import oracle
import psph
from helpers import (FLOAT_FIELDS_1D, FLOAT_FIELDS_3D, REL_TOL_FP64, compare, rel_l1, small_plume_config, sod_config)

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu] {msg}", flush=True)
    sys.stdout.flush()


def plume(reals, h_spread=0.0, **cfg_set):
    """A small plume of which only the first `reals` real particles (in read
    order) stay real; the others become pressure ghosts."""
    cfg = small_plume_config(half=400.0, top=800.0, sml_update_int=0)
    for k, v in cfg_set.items():
        setattr(cfg, k, v)
    P = psph.gen_plume(cfg, psph.meteo_standard(), 7, 0.01)
    real = np.nonzero(P["bc"] == 100)[0]
    P["bc"][real[reals:]] = 1
    rng = np.random.default_rng(reals)
    for k in ("vx", "vy", "vz", "svx", "svy", "svz"):
        P[k][real] = rng.standard_normal(len(real))
    P["h"][real] *= 1.3 * (1.0 + h_spread * rng.uniform(-1.0, 1.0, len(real)))
    P["phase"][real[::3]] = 2
    return cfg, P


CASES = {
    "1 target": dict(reals=1),
    "8 targets": dict(reals=8),
    "9 targets": dict(reals=9),
    "33 targets": dict(reals=33),
    "all": dict(reals=10**9),
    "h spread": dict(reals=10**9, h_spread=0.3),
    "list inside kernel box": dict(reals=10**9, h_spread=0.2, list_factor=2.0),
    "support inside kernel box": dict(reals=10**9, h_spread=0.2, cutoff2=1.5),
    "no filter, no smoothing": dict(reals=200, lans=0, energy_smooth=0),
    "smoothing ratio 3, all ghosts": dict(reals=200, e_smooth_ratio=3.0, pghost_contrib=2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_fp64_step_equals_oracle(name):
    cfg, P = plume(**CASES[name])
    S = oracle.State(cfg, P)
    with psph.Solver(cfg, len(P) + 20000) as G:
        G.load(P)
        for _ in range(2):
            S.step()
            G.step()
        errs = compare(G.read(), S.particles(), FLOAT_FIELDS_3D, REL_TOL_FP64)
    say(f"{name}: {len(P)} particles, max rel err {max(errs.values()):.2e}")


@pytest.mark.parametrize("form", ["pair", "exp", "pure"])
@pytest.mark.parametrize("name", ["9 targets", "list inside kernel box", "smoothing ratio 3, all ghosts"])
def test_fp32_forms_follow_fp64(name, form):
    out = {}
    for f, prec in (("fp64", psph.PSPH_FP64),
                    (form, dict(pair=psph.PSPH_FP32_PAIR, exp=psph.PSPH_FP32_EXP, pure=psph.PSPH_FP32_PURE)[form])):
        cfg, P = plume(**CASES[name])
        cfg.precision = prec
        with psph.Solver(cfg, len(P) + 20000) as G:
            G.load(P)
            pairs = G.step().n_pairs
            out[f] = (pairs, G.read())
    assert out["fp64"][0] == out[form][0] > 0
    for k in ("vx", "vy", "vz", "svx", "rho", "e", "p", "xi"):
        assert rel_l1(out[form][1][k], out["fp64"][1][k]) < 1e-5, k
    say(f"{name}, {form}: {out[form][0]} pairs as in FP64")


@pytest.mark.parametrize("n_left", [40, 203])
def test_1d_step_equals_oracle(n_left):
    cfg = sod_config(n_left)
    P = psph.gen_shock_tube(cfg, (1.0, 1.0, 0.0), (0.125, 0.1, 0.0), 0.0, 40, 20, 35, True)
    S = oracle.State(cfg, P)
    with psph.Solver(cfg, len(P) + 16) as G:
        G.load(P)
        for _ in range(3):
            S.step()
            G.step()
        compare(G.read(), S.particles(), FLOAT_FIELDS_1D, REL_TOL_FP64)
    say(f"Sod {n_left}: equal")



@pytest.mark.parametrize("form", ["fp64", "exp"])
@pytest.mark.parametrize("name", ["1 target", "9 targets", "33 targets", "h spread", "list inside kernel box",
                                  "support inside kernel box"])
def test_adaptive_h_equals_oracle(name, form):
    """An adaptation of three iterations, of which the converged targets leave
    the later ones; the FP32-exp form's exponential moves h by ~1e-9."""
    cfg, P = plume(**CASES[name])
    cfg.num_loop = 3
    if form == "exp":
        cfg.precision = psph.PSPH_FP32_EXP
    S = oracle.State(cfg, P)
    S.neighbors()
    S.adaptive_sml()
    with psph.Solver(cfg, len(P)) as G:
        G.load(P)
        G.search_neighs_consth()
        G.adaptive_sml()
        h = G.read()["h"]
    hs = S.particles()["h"]
    err = float(np.max(np.abs(h - hs) / hs))
    say(f"{name}, {form}: {int((hs != P['h']).sum())} adapted, max rel err of h {err:.2e}")
    assert err < (REL_TOL_FP64 if form == "fp64" else 1e-7)
