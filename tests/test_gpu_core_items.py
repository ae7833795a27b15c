"""Long rows of a dense core whose degree bound the caller chose: items at both
ends of the list (a piece per 2048 targets, and one item per candidate row)."""
import numpy as np
import pytest

import trust_amd as T

pytestmark = pytest.mark.gpu


def layers(a, h, t):
    """a rows over h + t vertices (every H, the first t of T), h rows over all
    h vertices of T: a * h * t triangles, all of them by edges A -> H."""
    H, Tv = a + np.arange(h), a + h + np.arange(h)
    adj = np.concatenate([np.tile(np.concatenate([H, Tv[:t]]), a), np.tile(Tv, h)]).astype(np.int32)
    deg = np.concatenate([np.full(a, h + t), np.full(h, h), np.zeros(h, np.int64)])
    return np.concatenate([[0], np.cumsum(deg)]), adj


@pytest.mark.parametrize("bound", [1025, 2048, 2101])
def test_long_rows_past_the_bound(gpu, bound):
    a, h, t = 6000, 2101, 100  # odd row lengths: every column is in the in-degree sample
    print(f"[gpu] core items, bound {bound}", flush=True)
    beg, adj = layers(a, h, t)
    with T.Context(gpu) as c:
        c.load(beg, adj)
        for _ in range(2):
            r = c.count(flags=T.FLAG_SHORT_WALK | T.FLAG_FRESH_INDEX, core_vertices=4096, core_min_degree=bound)
            assert r.triangles == a * h * t
            assert (r.dense_edges, r.dense_probes, r.probes) == (a * h, a * h * h, 0)
