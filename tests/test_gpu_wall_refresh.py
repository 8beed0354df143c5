"""The wall-ghost refresh against the oracle, where its work is split.

Ghosts are taken 8 consecutive particles at a time; two waves share the tiles
within reach of their images, which they list 64 rows of cells and 64 tiles at
a time.  The cases: a narrow and a wide ground (a group that spans two layers
of cells then has more than 64 rows), few particles, ghosts whose count leaves
groups partly filled, smoothing lengths that differ, support boxes inside the
kernel box, candidates that do not contribute.  Bar: the FP64 parity bar (1e-10
relative), every field; integers equal.
"""
import sys

import numpy as np
import pytest

import oracle
import psph
from helpers import FLOAT_FIELDS_3D, REL_TOL_FP64, compare, small_plume_config

pytestmark = pytest.mark.gpu


def plume(half, top, drop=0, h_spread=0.0, erupting=0, **cfg_set):
    cfg = small_plume_config(half=half, top=top, sml_update_int=0)
    cfg.wall_bc = 1
    for k, v in cfg_set.items():
        setattr(cfg, k, v)
    P = psph.gen_plume(cfg, psph.meteo_standard(), 11, 0.01)
    rng = np.random.default_rng(int(half) + drop)
    for k in ("vx", "vy", "vz", "xi"):
        P[k][:] = 0.1 * rng.standard_normal(len(P))
    P["h"][:] *= 1.0 + h_spread * rng.uniform(-1.0, 1.0, len(P))
    walls = np.nonzero(P["bc"] == 2)[0]
    P["bc"][walls[rng.permutation(len(walls))[:drop]]] = 1          # some wall ghosts contribute instead
    real = np.nonzero(P["bc"] == 100)[0]
    P["bc"][real[rng.permutation(len(real))[:erupting]]] = 0        # some particles contribute nothing
    return cfg, P


CASES = {
    "narrow": dict(half=300.0, top=300.0),
    "narrow, odd groups": dict(half=300.0, top=300.0, drop=37),
    "wide": dict(half=2600.0, top=400.0),
    "wide, h spread": dict(half=2600.0, top=400.0, drop=501, h_spread=0.25),
    "no contributor near": dict(half=300.0, top=300.0, erupting=10**9),
    "support inside kernel box": dict(half=500.0, top=500.0, h_spread=0.2, cutoff2=1.5),
}


@pytest.mark.parametrize("name", list(CASES))
def test_refresh_equals_oracle(name):
    cfg, P = plume(**CASES[name])
    S = oracle.State(cfg, P)
    S.apply_bcond()
    with psph.Solver(cfg, len(P)) as G:
        G.load(P)
        G.apply_bcond()
        Q = G.read()
    W = S.particles()
    walls = W["bc"] == 2
    changed = int((W["rho"][walls] != P["rho"][walls]).sum())
    errs = compare(Q, W, FLOAT_FIELDS_3D, REL_TOL_FP64)
    print(f"[gpu] {name}: {len(P)} particles, {changed} refreshed, max rel err {max(errs.values()):.2e}", flush=True)
    sys.stdout.flush()
