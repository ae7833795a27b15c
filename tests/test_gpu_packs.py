"""Packs of the wave tier: several short rows counted by one wave.

The edges of the rule: rows whose entries fill a pack exactly or overrun it by
one, ids on both sides of a power of two (the bits left for a row's number),
tables too small for a pack, and a pack whose insertion fails."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu

# out-degrees of consecutive rows (a pack holds 64 entries)
SHAPES = {
    "twos": [2] * 200,
    "exact": [32, 32, 16, 48, 63, 2, 64, 2, 62],
    "over": [33, 32, 65, 2, 64, 64, 3, 61, 1, 63, 2],
    "mixed": [2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37, 41] * 7,
    "ones and empties": [0, 1, 2, 0, 1, 3, 0, 0, 4, 1] * 12,
}


def rows_graph(degrees, ids, seed):
    """An oriented CSR over `ids` vertices: row r of the given out-degree over
    a window of later ids, dense enough to close triangles."""
    rng = np.random.default_rng(seed)
    n = len(degrees)
    lists = []
    for r in range(n):
        hi = min(ids, r + 1 + 3 * max(degrees) + 8)
        near = rng.permutation(np.arange(r + 1, hi))[:degrees[r]]
        # one entry in three far away: high ids, and every row of the pack may share them
        far = np.arange(ids - len(near), ids)
        take = (rng.random(len(near)) < 0.3) & (far > r)
        lists.append(np.unique(np.where(take, far, near)))
    beg = np.zeros(ids + 1, np.int64)
    beg[1:n + 1] = np.cumsum([len(x) for x in lists])
    beg[n + 1:] = beg[n]
    adj = np.concatenate(lists).astype(np.int32)
    T.validate(beg, adj)
    return beg, adj


@pytest.mark.parametrize("ids", [1 << 12, (1 << 12) + 1, 1 << 20, (1 << 24) - 1])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_packs_match_oracle(gpu, shape, ids):
    print(f"[gpu] packs {shape}, {ids} ids", flush=True)
    beg, adj = rows_graph(SHAPES[shape], ids, seed=ids % 97)
    want, probes = oracle.count_merge(beg, adj), oracle.probes(beg, adj)
    for load in (0, T.FLAG_OFFSETS64):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            for kw in (dict(chunk=64), dict(chunk=3), dict(chunk=64, wave_slots=128), dict(chunk=64, wave_slots=64),
                       dict(chunk=64, flags=T.FLAG_REFERENCE_WALK | T.FLAG_OFFSET_LOOKUP),
                       dict(chunk=64, threads=64, blocks=1), dict(chunk=64, flags=T.FLAG_WAVE_ONLY)):
                flags = kw.pop("flags", T.FLAG_REFERENCE_WALK)
                r = c.count(flags=flags, **kw)
                assert (r.triangles, r.probes) == (want, probes), (load, kw, flags)
            r = c.count(flags=T.FLAG_SHORT_WALK, chunk=64, core_vertices=-1)
            assert (r.triangles, r.probes) == (want, oracle.probes_short(beg, adj)), load
            share = [c.count(flags=T.FLAG_REFERENCE_WALK, chunk=2, rank=k, total_process=3) for k in range(3)]
            assert sum(r.triangles for r in share) == want


def test_pack_of_colliding_keys_is_counted_by_vertex(gpu):
    # row j holds c - 0x9E5 j: the keys of all rows share both buckets, four
    # slots for eight keys, so the pack's insertion fails
    c, rows = 60000, 8
    edges = []
    for j in range(rows):
        key, other = c - 0x9E5 * j, c + 1 + j
        edges += [(j, key), (j, other), (key, other)]
    V = c + 1 + rows
    e = np.array(sorted(edges))
    beg = np.zeros(V + 1, np.int64)
    np.add.at(beg, e[:, 0] + 1, 1)
    beg, adj = np.cumsum(beg), e[:, 1].astype(np.int32)
    assert oracle.count_merge(beg, adj) == rows
    r = T.count_csr(beg, adj, chunk=64, flags=T.FLAG_REFERENCE_WALK, device=gpu)
    assert (r.triangles, r.probes) == (rows, oracle.probes(beg, adj))


def test_packs_stay_in_their_graph(gpu):
    rng = np.random.default_rng(4)
    parts, vbase, ebase = [], [0], 0
    for k in range(60):
        b, a = rows_graph([int(x) for x in rng.integers(0, 9, 5 + k % 7)], 64, seed=k)
        parts.append((b, a))
        vbase.append(vbase[-1] + 64)
    beg = np.concatenate([[0]] + [np.diff(b) for b, _ in parts]).cumsum()
    adj = np.concatenate([a + 64 * k for k, (_, a) in enumerate(parts)]).astype(np.int32)
    want = [oracle.count_merge(b, a) for b, a in parts]
    assert sum(want) > 0
    with T.Context(gpu) as c:
        c.load_batch(beg, adj, np.array(vbase))
        for kw in (dict(chunk=64), dict(chunk=64, flags=T.FLAG_HIP_GRAPH), dict(chunk=64, flags=T.FLAG_HIP_GRAPH), dict()):
            counts, _, r = c.count_batch(**kw)
            assert counts.tolist() == want, kw
            assert r.probes == oracle.probes(beg, adj)
