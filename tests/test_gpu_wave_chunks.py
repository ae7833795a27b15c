"""The wave tier's chunks: the parts beyond a vertex's first, then the first
quarter of the vertices in small chunks, then the others.

With one workgroup of one wave the first quarter is taken in chunks of more
than one vertex from 32 vertices on; the sizes stand around multiples of that,
of the quarter and of the 64-vertex chunk."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


def rows_graph(n, longest, seed):
    """n rows in descending length (2 to longest) over n + 130 later ids."""
    rng = np.random.default_rng(seed)
    m = n + 130
    deg = np.maximum(2, longest - (longest - 2) * np.arange(n) // max(n // 2, 1))
    lists = [np.sort(i + 1 + rng.permutation(min(m - i - 1, 120))[:d]) for i, d in enumerate(deg)]
    lists += [np.zeros(0, np.int64)] * (m - n)
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    T.validate(beg, adj)
    return beg, adj


@pytest.mark.parametrize("n", [1, 3, 4, 31, 32, 33, 127, 128, 129, 255, 257, 1023, 1025, 4099])
@pytest.mark.parametrize("longest", [64, 65, 100])  # to 64: all chunks alike
def test_chunks_match_oracle(gpu, n, longest):
    print(f"[gpu] wave chunks {n} {longest}", flush=True)
    beg, adj = rows_graph(n, longest, n)
    want = oracle.count_merge(beg, adj)
    for load in (0, T.FLAG_OFFSETS64):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            for walk, probes in ((T.FLAG_REFERENCE_WALK, oracle.probes(beg, adj)),
                                 (T.FLAG_SHORT_WALK, oracle.probes_short(beg, adj))):
                for kw in (dict(), dict(threads=64, blocks=1), dict(threads=256, blocks=2), dict(chunk=5)):
                    for ranks in (1, 2, 5):
                        r = [c.count(flags=walk, core_vertices=-1, rank=k, total_process=ranks, **kw)
                             for k in range(ranks)]
                        got = sum(x.triangles for x in r), sum(x.probes for x in r)
                        assert got == (want, probes), (load, walk, kw, ranks)
