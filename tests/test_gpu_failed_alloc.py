"""A device allocation that fails is one call's error, not the next call's."""
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["resident", "fresh", "one-shot", "tiles", "batch"])
def test_next_call_counts(gpu, call):
    print(f"[gpu] {call} after a failed allocation", flush=True)
    beg, adj = T.rmat_csr(10, 8, seed=1)
    want = oracle.count_merge(beg, adj)
    tiles = T.partition_csr(beg, adj, 2)
    with T.Context(gpu) as c:
        if call == "batch":
            c.load_batch(beg, adj, [0, len(beg) - 1])
        else:
            c.load(beg, adj)
        count = {"resident": lambda: c.count().triangles,
                 "fresh": lambda: c.count(flags=T.FLAG_FRESH_INDEX).triangles,
                 "one-shot": lambda: T.count_csr(beg, adj).triangles,
                 "tiles": lambda: T.count_tiles(tiles, 2).triangles,
                 "batch": lambda: c.count_batch()[2].triangles}[call]
        assert count() == want
        for _ in range(2):
            with pytest.raises(T.TrustError) as e:
                T.membench_copy(1 << 50)  # more than any device has
            assert e.value.code == T.ERR_OOM
            assert count() == want
