"""Shares of one count by ranks that each build a walk index of their own.

The entries of a walk row come in another order with every build, so a vertex
is one rank's as a whole where its walk is a built index."""
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [12, 16])
@pytest.mark.parametrize("P", [2, 3])
def test_each_rank_with_its_own_context(gpu, scale, P):
    print(f"[gpu] {P} ranks, rmat{scale}", flush=True)
    beg, adj = T.rmat_csr(scale, 16, seed=1)
    want = oracle.count_hash(beg, adj)
    for walk, probes in ((T.FLAG_SHORT_WALK, oracle.probes_short(beg, adj)),
                         (T.FLAG_REFERENCE_WALK, oracle.probes(beg, adj))):
        for load in (0, T.FLAG_OFFSETS64):
            r = []
            for k in range(P):
                with T.Context(gpu) as c:
                    c.load(beg, adj, load)
                    r.append(c.count(flags=walk, rank=k, total_process=P))
            assert (sum(x.triangles for x in r), sum(x.probes for x in r)) == (want, probes), (walk, load)
        r = [T.count_csr(beg, adj, flags=walk, rank=k, total_process=P) for k in range(P)]
        assert (sum(x.triangles for x in r), sum(x.probes for x in r)) == (want, probes), walk


@pytest.mark.parametrize("n", [1, 2])
def test_tiles(gpu, n):
    print(f"[gpu] ranks over {n}x{n} tiles", flush=True)
    beg, adj = T.rmat_csr(14, 16, seed=1)
    want = oracle.count_hash(beg, adj)
    tiles = T.partition_csr(beg, adj, n)
    for walk in (0, T.FLAG_REFERENCE_WALK):
        r = [T.count_tiles(tiles, n, flags=walk, rank=k, total_process=3) for k in range(3)]
        assert sum(x.triangles for x in r) == want, walk
