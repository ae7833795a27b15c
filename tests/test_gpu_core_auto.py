"""The automatic dense core and the degree bound that follows its size."""
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offsets64", [False, True])
def test_automatic_core_rmat20(gpu, offsets64):
    # enough edges for the automatic core, sources enough for several items a grab
    print(f"[gpu] automatic core, rmat20, offsets64={offsets64}", flush=True)
    beg, adj = T.rmat_csr(20, 16, seed=2)
    want, short = oracle.count_hash(beg, adj), oracle.probes_short(beg, adj)
    with T.Context(gpu) as c:
        c.load(beg, adj, T.FLAG_OFFSETS64 if offsets64 else 0)
        for kw in (dict(flags=T.FLAG_SHORT_WALK), dict(flags=T.FLAG_SHORT_WALK | T.FLAG_FRESH_INDEX),
                   dict(flags=T.FLAG_SHORT_WALK, core_vertices=4096), dict(flags=T.FLAG_SHORT_WALK, core_vertices=512),
                   dict(flags=T.FLAG_SHORT_WALK, core_min_degree=40), dict(flags=T.FLAG_SHORT_WALK)):
            r = c.count(**kw)
            assert r.triangles == want, kw
            assert r.core_vertices > 0 and r.dense_edges > 0, kw
            assert r.probes + r.dense_probes == short, kw
        assert c.count(flags=T.FLAG_SHORT_WALK, core_vertices=-1).probes == short


@pytest.mark.parametrize("K", [256, 1024, 16384])
def test_core_bound_by_its_size(gpu, K):
    # core_min_degree 0: a 48th of the core, at least 64, which rmat16's core has above it
    beg, adj = T.rmat_csr(16, 16, seed=1)
    want, short = oracle.count_hash(beg, adj), oracle.probes_short(beg, adj)
    with T.Context(gpu) as c:
        c.load(beg, adj)
        for _ in range(2):
            r = c.count(flags=T.FLAG_SHORT_WALK | T.FLAG_FRESH_INDEX, core_vertices=K)
            assert r.triangles == want
            assert r.probes + r.dense_probes == short
