"""The passes over the CSR that a fresh count makes: both walks' totals, the
walk they decide, the start index and the cost features, at row counts around
the groups that a wave takes (8 to 64 rows) and with long rows among short ones."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def graph(V, longest, seed):
    """Rows of 0 to 6 later vertices and, every 9th row, of up to `longest`."""
    rng = np.random.default_rng(seed)
    lists = []
    for r in range(V):
        want = int(rng.integers(0, 7)) if r % 9 else longest
        room = V - 1 - r
        lists.append(np.sort(r + 1 + rng.permutation(room)[:min(want, room)]))
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    T.validate(beg, adj)
    return beg, adj


@pytest.mark.parametrize("longest", [8, 300])
@pytest.mark.parametrize("V", [2, 7, 8, 9, 63, 64, 65, 127, 129, 1000, 2049])
def test_fresh_count_totals_and_features(gpu, V, longest):
    print(f"[gpu] index passes V={V} longest={longest}", flush=True)
    beg, adj = graph(V, longest, seed=V)
    want = oracle.count_merge(beg, adj)
    ref, short = oracle.probes(beg, adj), oracle.probes_short(beg, adj)
    for load in (0, T.FLAG_OFFSETS64):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            for flags in (0, T.FLAG_FRESH_INDEX, T.FLAG_FRESH_INDEX | T.FLAG_OFFSET_LOOKUP, T.FLAG_SHORT_WALK,
                          T.FLAG_REFERENCE_WALK, 0, T.FLAG_FRESH_INDEX | T.FLAG_SHORT_WALK):
                r = c.count(flags=flags)
                side = bool(flags & T.FLAG_SHORT_WALK) or (not flags & T.FLAG_REFERENCE_WALK and short <= 0.45 * ref)
                assert r.walk_used == int(side), flags
                assert (r.triangles, r.probes) == (want, short if side else ref), flags
            assert np.allclose(c.features(), oracle.mlp_scaled_features(beg, adj), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("seed", [1, 2])
def test_short_side_after_the_reference_pass(gpu, seed):
    # a flat degree distribution (the reference pass goes first) whose probes
    # the short side more than halves: every second row points at long rows
    rng = np.random.default_rng(seed)
    n, d = 400, 40
    lists = [np.sort(np.append(2 * n + rng.permutation(n)[:2], 3 * n + rng.integers(200))) for _ in range(2 * n)]
    lists += [3 * n + np.sort(rng.permutation(200)[:d]) for _ in range(n)]
    lists += [np.zeros(0, np.int64)] * 200
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    T.validate(beg, adj)
    ref, short = oracle.probes(beg, adj), oracle.probes_short(beg, adj)
    assert short <= 0.45 * ref and np.diff(beg).max() * (len(beg) - 1) < 24 * len(adj)
    want = oracle.count_merge(beg, adj)
    assert want > 0
    with T.Context(gpu) as c:
        c.load(beg, adj)
        for flags in (0, T.FLAG_REFERENCE_WALK, T.FLAG_FRESH_INDEX, 0, T.FLAG_REFERENCE_WALK):
            r = c.count(flags=flags)
            side = not flags & T.FLAG_REFERENCE_WALK
            assert (r.walk_used, r.triangles, r.probes) == (int(side), want, short if side else ref), flags
