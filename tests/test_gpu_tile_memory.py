"""Tile streams under a device-memory cap: whatever cap a stream with 2n + 2
slots fits, the default stream, which keeps all tiles where it can, fits too."""
import numpy as np
import pytest

import oracle
import trust_amd as T

pytestmark = pytest.mark.gpu
N = 4


def uneven(tiles, n):
    """The tiles with rows of no entries after each class's, so that every slot
    is larger than most tiles need."""
    out = []
    for k, (b, a) in enumerate(tiles):
        extra = 200_000 if k // n == n - 1 else 0
        out.append((np.concatenate([b, np.full(extra, b[-1])]), a))
    return out


@pytest.mark.parametrize("shape", ["even", "uneven"])
def test_default_fits_where_few_slots_do(gpu, shape, tmp_path):
    beg, adj = T.rmat_csr(18, 16, seed=1)
    want = oracle.count_hash(beg, adj)
    tiles = T.partition_csr(beg, adj, N)
    if shape == "uneven":
        tiles = uneven(tiles, N)
    held = T.device_memory_held()

    def count(cap, **kw):
        T.set_device_memory_cap(held + cap)
        try:
            return T.count_tiles(tiles, N, **kw).triangles
        except T.TrustError as e:
            assert e.code == T.ERR_OOM, e
            return None

    try:
        fits, least = [], None
        for cap in range(4 << 20, 100 << 20, 2 << 20):
            few = count(cap, reserved=[2 * N + 2, 0, 0])
            assert few in (None, want), cap
            got = count(cap)
            print(f"[gpu] {shape} cap {cap >> 20} MB: {few} with few slots, {got} by default", flush=True)
            assert got == few, cap
            fits.append(few is not None)
            if few is not None and least is None:
                least = cap
        assert fits == sorted(fits) and True in fits and False in fits
        # a journal under the least cap: only the jobs asked for, then the rest
        T.set_device_memory_cap(held + least)
        journal = str(tmp_path / "journal")
        missing, _, _ = T.count_tiles_journal(tiles, N, journal, max_new_jobs=10)
        assert missing == N ** 3 - 10
        missing, r, jobs = T.count_tiles_journal(tiles, N, journal)
        assert (missing, r.triangles, int(jobs.sum())) == (0, want, want)
        T.set_device_memory_cap(0)
        assert T.count_tiles(tiles, N).triangles == want
        assert T.device_memory_held() == held
    finally:
        T.set_device_memory_cap(0)


def test_many_jobs_need_no_block_each(gpu, tmp_path):
    # 512 jobs of two counts: with a control block kept for each the stream takes 21 MB
    n = 8
    beg, adj = T.rmat_csr(18, 16, seed=1)
    want = oracle.count_hash(beg, adj)
    tiles = T.partition_csr(beg, adj, n)
    print("[gpu] 8 x 8 tiles under 13 MB", flush=True)
    try:
        T.set_device_memory_cap(T.device_memory_held() + (13 << 20))
        assert T.count_tiles(tiles, n).triangles == want
        for jobs in (1, 15, 16, 17):  # around the control blocks' ring
            journal = str(tmp_path / f"journal{jobs}")
            missing, _, _ = T.count_tiles_journal(tiles, n, journal, max_new_jobs=jobs)
            assert missing == n ** 3 - jobs
            missing, r, each = T.count_tiles_journal(tiles, n, journal)
            assert (missing, r.triangles, int(each.sum())) == (0, want, want)
    finally:
        T.set_device_memory_cap(0)
