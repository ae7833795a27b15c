"""Tiles are checked once each, with the verdicts of the job-by-job check."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def bad(tiles, n, kind):
    tiles = [(b.copy(), a.copy()) for b, a in tiles]
    t = n + 1 if n > 1 else 0  # tile (1, 1)
    b, a = tiles[t]
    if kind == "negative id":
        a[len(a) // 2] = -5
    elif kind == "id past the probe tile's rows":
        a[len(a) // 2] = len(tiles[(t % n) * n][0]) - 1
    elif kind == "decreasing offsets":
        b[2], b[3] = b[3] + 1, b[2]
    elif kind == "offsets short of the entries":
        b[-1] -= 1
    elif kind == "first offset":
        b[0] = 1
    else:  # a row more than the other tiles of its class
        b = np.append(b, b[-1])
    tiles[t] = (b, a)
    return tiles


@pytest.mark.parametrize("kind", ["negative id", "id past the probe tile's rows", "decreasing offsets",
                                  "offsets short of the entries", "first offset", "a row too many"])
@pytest.mark.parametrize("n", [2, 3])
def test_bad_tiles_are_refused(gpu, n, kind):
    beg, adj = T.rmat_csr(10, 8, seed=1)
    tiles = T.partition_csr(beg, adj, n)
    print(f"[gpu] bad tiles n={n}: {kind}", flush=True)
    with pytest.raises(T.TrustError) as e:
        T.count_tiles(bad(tiles, n, kind), n)
    assert e.value.code == T.ERR_FORMAT
    assert T.count_tiles(tiles, n).triangles == oracle.count_merge(beg, adj)


@pytest.mark.parametrize("slots", [0, 3, 5, 16, 100])
@pytest.mark.parametrize("n", [1, 2, 4])
def test_every_number_of_slots_counts_the_same(gpu, n, slots):
    beg, adj = T.rmat_csr(12, 8, seed=2)
    want = oracle.count_merge(beg, adj)
    tiles = T.partition_csr(beg, adj, n)
    for flags in (0, T.FLAG_REFERENCE_WALK, T.FLAG_NO_VALIDATE, T.FLAG_OFFSETS64):
        r = T.count_tiles(tiles, n, flags=flags, reserved=[slots, 0, 0])
        assert r.triangles == want, (n, slots, flags)
