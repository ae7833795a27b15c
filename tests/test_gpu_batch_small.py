"""Small batches, dealt out without a queue: sizes around one and two vertices
per wave of one workgroup, and around the bounds of 8 and 32."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("longest", [30, 100])  # above 64 the bound is 8 vertices a wave
@pytest.mark.parametrize("sizes", [[1, 2, 3], [4, 4], [31, 33], [64, 65, 127], [500, 3, 520]], ids=str)
def test_small_batches(gpu, sizes, longest):
    print(f"[gpu] small batch {sizes} {longest}", flush=True)
    rng = np.random.default_rng(sum(sizes))
    lists, vbase, want = [], [0], []
    for n in sizes:
        m = n + 2 * longest
        g = [np.sort(i + 1 + rng.permutation(m - i - 1)[: 2 + rng.integers(0, longest - 1)]) for i in range(n)]
        g += [np.zeros(0, np.int64)] * (m - n)
        b = np.concatenate([[0], np.cumsum([len(x) for x in g])])
        want.append(oracle.count_merge(b, np.concatenate(g).astype(np.int32)))
        lists += [x + vbase[-1] for x in g]
        vbase.append(vbase[-1] + m)
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    with T.Context(gpu) as c:
        c.load_batch(beg, adj, np.array(vbase))
        for kw in (dict(), dict(threads=64, blocks=1), dict(threads=256, blocks=1), dict(flags=T.FLAG_HIP_GRAPH)):
            for _ in range(2):
                got, _, r = c.count_batch(**kw)
                assert list(got) == want and r.triangles == sum(want), kw
