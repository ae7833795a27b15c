"""The learned schedule as a context's first count: its list is made before any
other plan has sized the list's buffer."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [60, 4000, 70000])
def test_learned_count_comes_first(gpu, n):
    print(f"[gpu] learned first {n}", flush=True)
    rng = np.random.default_rng(n)
    lists = [np.unique(i + 1 + rng.integers(0, 40, 2 + i % 30)) for i in range(n - 1)]
    lists = [x[x < n] for x in lists] + [np.zeros(0, np.int64)]
    beg = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    adj = np.concatenate(lists).astype(np.int32)
    want = oracle.count_merge(beg, adj)
    with T.Context(gpu) as c:
        c.load(beg, adj)
        c.train_cost_model(epochs=2, max_samples=1000, seed=1)
        model = c.get_cost_model()
    for load in (0, T.FLAG_OFFSETS64):
        with T.Context(gpu) as c:
            c.load(beg, adj, load)
            c.set_cost_model(model)
            for schedule in (T.SCHED_LEARNED, T.SCHED_DEGREE, T.SCHED_LEARNED):
                r = c.count(schedule=schedule)
                assert (r.triangles, r.schedule_used) == (want, schedule)
