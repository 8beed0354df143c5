"""The order in which the group passes take a cell's targets, at the edges of its
runs of 128 and halves of 64 to 8, against the oracle.

One cell holds every particle (list_all), so that the number of targets is the
length of the runs; without jitter most coordinates of the lattice are ties.  The
order decides only which targets share a group: every field keeps the parity bar
of the FP64 form (1e-10 relative).
"""
import pytest

import oracle
import psph
from helpers import FLOAT_FIELDS_3D, REL_TOL_FP64, compare
from test_gpu_group_passes import plume, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reals", [7, 8, 9, 17, 63, 64, 65, 127, 128, 129, 137, 300])
def test_runs_equal_oracle(reals):
    cfg, P = plume(reals, h_spread=0.2, list_all=1)
    if reals % 2:
        for k in "xyz":
            P[k][:] = (P[k] / (0.5 * cfg.h_air)).round() * (0.5 * cfg.h_air)
    S = oracle.State(cfg, P)
    with psph.Solver(cfg, len(P) + 2000) as G:
        G.load(P)
        S.step()
        G.step()
        errs = compare(G.read(), S.particles(), FLOAT_FIELDS_3D, REL_TOL_FP64)
    say(f"{reals} targets in one cell: max rel err {max(errs.values()):.2e}")
