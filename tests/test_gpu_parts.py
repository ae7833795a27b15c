"""Vertices of long walks, counted in parts by several workgroups.

A part is 128 walk entries at least (512 in the large-LDS launch, whose tables
start above 2048 neighbours here): walks one entry short of a part's end, at
it and past it, and runs of more parts than one wave looks back over at once."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def hubs_graph(degrees, seed=1):
    """One row of each out-degree over a shared set of later vertices that
    have two edges each among themselves."""
    rng = np.random.default_rng(seed)
    n, m = len(degrees), max(degrees) + 40
    lists = [np.sort(n + rng.permutation(m)[:d]) for d in degrees]
    lists += [n + np.unique(np.minimum(i + 1 + rng.integers(0, 30, 2), m - 1)) for i in range(m - 1)]
    lists = [x[x > r] for r, x in enumerate(lists)] + [np.zeros(0, np.int64)]
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    T.validate(beg, adj)
    return beg, adj


@pytest.mark.parametrize("degrees", [
    [127, 128, 129, 255, 256, 257], [512, 511, 513, 130, 101, 2047], [2048, 2049, 2100, 2560, 2561, 3000],
    [9000, 8192, 8193, 150], [40000, 129], [20000]], ids=lambda d: str(max(d)))
def test_parts_match_oracle(gpu, degrees):
    print(f"[gpu] parts {degrees}", flush=True)
    beg, adj = hubs_graph(degrees)
    want = oracle.count_merge(beg, adj)
    assert want > 0
    for load in (0, T.FLAG_OFFSETS64):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            for walk, probes in ((T.FLAG_REFERENCE_WALK, oracle.probes(beg, adj)),
                                 (T.FLAG_SHORT_WALK, oracle.probes_short(beg, adj))):
                for kw in (dict(), dict(threads=64), dict(threads=1024, blocks=3), dict(chunk=7),
                           dict(lds_budget=8192, threads=64, wave_slots=64)):
                    r = c.count(flags=walk, core_vertices=-1, **kw)
                    assert (r.triangles, r.probes) == (want, probes), (load, walk, kw)
                    assert r.n_spill + r.n_hub + r.n_wave <= len(beg) - 1
                share = [c.count(flags=walk, rank=k, total_process=3) for k in range(3)]
                assert sum(r.triangles for r in share) == want
            r = c.count(flags=T.FLAG_REFERENCE_WALK)
            assert r.n_spill + r.n_hub + r.n_wave == int((np.diff(beg) >= 2).sum())
            # each vertex's table is rebuilt in every part and counted once
            r = c.count(flags=T.FLAG_REFERENCE_WALK | T.FLAG_REBUILD_LINEAR)
            assert r.triangles == want
            assert r.linear_rebuilds == r.n_spill + r.n_hub + r.n_wave
