"""A step queues its passes and reads their errors once, at its end: what a failing
step reports and leaves behind is what the stages called one by one leave.

The adaptation queues its iterations behind the first likewise; where a later one
needs more memory for its lists than the first, it is made again (against the
oracle, 1e-10 relative).
"""
import numpy as np
import pytest

import oracle
import psph
from helpers import REL_TOL_FP64
from test_gpu_group_passes import plume, say

pytestmark = pytest.mark.gpu


def broken(stage):
    cfg, P = plume(10**9)
    real = np.nonzero(P["bc"] == 100)[0]
    if stage == "rhs":
        P["rho"][real[5]] = -1.0              # 1 / rho of a neighbour
    elif stage == "density":
        P["m"][:] = 0.0                       # no mass in the sums
    else:
        P["c"][real[5]] = 0.0
    return cfg, P


@pytest.mark.parametrize("stage", ["timestep", "rhs", "density"])
def test_failing_step(stage):
    cfg, P = broken(stage)
    got = {}
    for how in ("step", "stages"):
        with psph.Solver(cfg, len(P) + 2000) as G:
            G.load(P)
            with pytest.raises(psph.PsphError, match=stage):
                if how == "step":
                    G.step()
                else:
                    dt = G.timestep()
                    G.search_neighs_consth()
                    G.mom_engr_update(dt)
                    G.smooth_density()
            got[how] = G.read()
            # and the context goes on
            ok = plume(10**9)[1]
            G.load(ok)
            assert G.step().n_pairs > 0
    for k in ("x", "y", "z", "h", "m", "bc") + (("rho",) if stage != "density" else ()):
        assert np.array_equal(got["step"][k], got["stages"][k]), k
    say(f"{stage}: reported, state kept")


@pytest.mark.parametrize("scale", [0.3, 0.6])
def test_adaptation_outgrows_its_first_lists(scale):
    cfg, P = plume(10**9)
    cfg.num_loop = 6
    P["h"][P["bc"] == 100] *= scale
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
    say(f"h x {scale}: max rel err of h {err:.2e}")
    assert err < REL_TOL_FP64
