"""The walk of a default count depends on the graph and the core asked for,
not on the counts made before it."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def layers(a, h, t):
    """a rows over h + t vertices, h rows over the t: rows of like length, whose
    walk's two sides are alike and whose edges a core takes whole."""
    H, Tv = a + np.arange(h), a + h + np.arange(t)
    adj = np.concatenate([np.tile(np.concatenate([H, Tv]), a), np.tile(Tv, h)]).astype(np.int32)
    deg = np.concatenate([np.full(a, h + t), np.full(h, t), np.zeros(t, np.int64)])
    return np.concatenate([[0], np.cumsum(deg)]), adj


@pytest.mark.parametrize("offsets64", [False, True])
def test_default_walk_after_a_forced_one(gpu, offsets64):
    print(f"[gpu] walk choice, offsets64={offsets64}", flush=True)
    a, h, t = 1000, 151, 150
    beg, adj = layers(a, h, t)
    want, ref, short = a * h * t, oracle.probes(beg, adj), oracle.probes_short(beg, adj)
    assert short > 0.45 * ref
    core = dict(core_vertices=512, core_min_degree=64)
    load = T.FLAG_OFFSETS64 if offsets64 else 0
    for order in ("default first", "forced first"):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            if order == "default first":
                r = c.count(**core)
                assert (r.triangles, r.walk_used, r.probes) == (want, 0, ref)
            r = c.count(flags=T.FLAG_SHORT_WALK, **core)
            assert (r.triangles, r.walk_used, r.dense_edges) == (want, 1, a * h)
            for _ in range(2):
                r = c.count(**core)
                assert (r.triangles, r.walk_used, r.probes) == (want, 0, ref), order
