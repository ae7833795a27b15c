"""A graph with empty rows for ids that no edge names counts as without them:
same walk, same core, same probes."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def facts(r):
    return (r.triangles, r.walk_used, r.core_vertices, r.probes, r.dense_edges, r.dense_probes)


@pytest.mark.parametrize("scale,pairs,once", [(18, 48, False), (20, 16, False), (20, 30, True), (14, 16, False)])
@pytest.mark.parametrize("offsets64", [False, True])
def test_empty_rows_change_nothing(gpu, scale, pairs, once, offsets64):
    print(f"[gpu] padded rmat{scale}, {pairs} pairs, offsets64={offsets64}", flush=True)
    beg, adj = T.rmat_csr(scale, pairs, seed=3)
    V = len(beg) - 1
    padded = np.concatenate([beg, np.full(4 * (1 << scale) - V, beg[-1])])
    flags = T.FLAG_OFFSETS64 if offsets64 else 0

    def count(b):
        if once:
            return T.count_csr(b, adj, flags=flags)
        with T.Context(gpu) as c:
            c.load(b, adj, flags)
            return c.count()

    r, s = count(beg), count(padded)
    assert facts(r) == facts(s)
    assert (r.core_vertices > 0) == (scale > 14) and r.walk_used == int(scale > 14)
    assert (r.vertices, s.vertices) == (V, len(padded) - 1)
    assert r.probes + r.dense_probes == (oracle.probes_short if r.walk_used else oracle.probes)(beg, adj)
