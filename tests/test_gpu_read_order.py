"""psph_read's order, made on the GPU: THashTable order (slot, then key0, key1,
key2), ties in device order, removed particles left out.

Keys are random, from small sets so that every level has ties, and from the whole
range so that the slot's roundings count; the bar is equality.
"""
import numpy as np
import pytest

import psph
from helpers import small_plume_config, sod_config

pytestmark = pytest.mark.gpu


def slots(k0, k1, size, dim):
    if dim == 1:
        return k0.astype(np.int64)
    s2 = size // 10
    umax = 4294967295.0
    return ((k0 / umax * (size - s2)).astype(np.int32) + (k1 / umax * s2).astype(np.int32)).astype(np.int64)


@pytest.mark.parametrize("dim", [1, 3])
@pytest.mark.parametrize("n", [1, 2, 64, 65, 1023, 20001])
def test_order_equals_lexsort(n, dim):
    cfg = small_plume_config() if dim == 3 else sod_config(40)
    rng = np.random.default_rng(n)
    P = psph.Particles(n)
    for k in P.a:
        P[k][:] = rng.uniform(1.0, 2.0, n) if P[k].dtype.kind == "f" else np.arange(n) % 7
    few = np.array([0, 1, 7, 2**31 - 1, 2**31, 2**32 - 2, 2**32 - 1], np.uint32)
    for k in ("key0", "key1", "key2"):
        pick = rng.uniform(size=n) < 0.5
        P[k][:] = np.where(pick, rng.choice(few, n), rng.integers(0, 2**32, n, dtype=np.uint32))
    P["bc"][:] = rng.choice([-1, 0, 1, 2, 100], n)
    live = np.nonzero(P["bc"] >= 0)[0]
    k0, k1, k2 = (P[k][live] for k in ("key0", "key1", "key2"))
    want = live[np.lexsort((k2, k1, k0, slots(k0.astype(np.float64), k1.astype(np.float64), cfg.p_table_size, dim)
                            if dim == 3 else k0))]
    with psph.Solver(cfg, n + 8) as G:
        G.load(P)
        assert G.count() == (len(live), int((P["bc"] == 100).sum()))
        Q = G.read()
        R = G.read()                      # and the state it read is untouched
    assert len(Q) == len(live)
    for k in P.a:
        assert np.array_equal(Q[k], P[k][want]), k
        assert np.array_equal(R[k], Q[k]), k
