"""Dense graphs take the short-side walk when the dense core leaves little of
it; a count without the core, or a rank's share, keeps the reference walk."""
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offsets64", [False, True])
def test_dense_graph_takes_the_core(gpu, offsets64):
    print(f"[gpu] dense rmat18, offsets64={offsets64}", flush=True)
    beg, adj = T.rmat_csr(18, 48, seed=3)
    want, ref, short = oracle.count_hash(beg, adj), oracle.probes(beg, adj), oracle.probes_short(beg, adj)
    with T.Context(gpu) as c:
        c.load(beg, adj, T.FLAG_OFFSETS64 if offsets64 else 0)
        for kw in (dict(), dict(core_vertices=-1), dict(flags=T.FLAG_FRESH_INDEX), dict()):
            r = c.count(**kw)
            assert (r.triangles, r.walk_used) == (want, int("core_vertices" not in kw)), kw
            assert r.probes + r.dense_probes == (short if r.walk_used else ref), kw
        share = [c.count(rank=k, total_process=2) for k in range(2)]
        assert sum(r.triangles for r in share) == want and {r.walk_used for r in share} == {0}


def test_one_shot_leaves_a_small_core_out(gpu):
    beg, adj = T.rmat_csr(18, 48, seed=3)
    r = T.count_csr(beg, adj)
    assert (r.triangles, r.core_vertices) == (oracle.count_hash(beg, adj), 0)
