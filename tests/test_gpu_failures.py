"""Failure paths of the C ABI on the GPU: oversize requests and device
allocation failures (forced through the test-support option "fail_alloc",
which makes the n-th allocation of this thread report out-of-memory).

Every failed call must return its status without side effects -- an add
that fails stores nothing -- and the same index must then give the oracle's
results (index_flat.dart:62-137 for search and range search, kmeans.dart:91-140
for the k-means step)."""
import numpy as np
import pytest

import oracle
from _parity import assert_knn_parity, assert_range_parity
from vector_store import synthetic as syn

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()


def _oom(vs, fn):
    with pytest.raises(vs.VsError) as e:
        fn()
    assert e.value.code == vs._native.VS_ERR_OOM, str(e.value)


def test_oversize_reserve(vs):
    """More rows than int32 ids can name is invalid; a representable but
    impossible reservation (2^31 - 1 rows of 16 KiB) is out of memory; the
    index stays usable."""
    idx = vs.GpuIndexFlat.l2(4096, storage="f32")
    with pytest.raises(ValueError, match="int32"):
        idx.reserve(1 << 31)
    _oom(vs, lambda: idx.reserve((1 << 31) - 1))
    xb = syn.int_grid(300, 4096, 1, 0)
    xq = syn.int_grid(4, 4096, 1, 1)
    idx.add(xb)
    r = idx.search(xq, 5)
    idx.close()
    Dr, Ir = oracle.flat_search(xb, xq, 5, 0, NT)
    assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)


def test_add_allocation_failure_stores_nothing(vs):
    xb = syn.int_grid(2000, 64, 2, 0)
    idx = vs.GpuIndexFlat.l2(64)
    idx.set_option("fail_alloc", 1)
    _oom(vs, lambda: idx.add(xb))
    idx.set_option("fail_alloc", 0)
    assert idx.ntotal == 0
    idx.add(xb)
    assert idx.ntotal == 2000
    xq = syn.int_grid(7, 64, 2, 1)
    r = idx.search(xq, 10)
    idx.close()
    Dr, Ir = oracle.flat_search(xb, xq, 10, 0, NT)
    assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)


@pytest.mark.parametrize("nq", [5, 600])
def test_search_allocation_failures(vs, nq):
    """The first search of an index allocates its scratch; the n-th of those
    allocations fails for n = 1, 2, ...: each failed search reports
    out-of-memory, and the next one, with nothing forced, is exact."""
    xb = syn.int_grid(5000, 128, 3, 0)
    xq = syn.int_grid(nq, 128, 3, 1)
    Dr, Ir = oracle.flat_search(xb, xq, 20, 0, NT)
    failed = 0
    for n in range(1, 12):
        idx = vs.GpuIndexFlat.l2(128)
        idx.add(xb)
        idx.set_option("fail_alloc", n)
        try:
            idx.search(xq, 20)
        except vs.VsError as e:
            assert e.code == vs._native.VS_ERR_OOM
            failed += 1
        idx.set_option("fail_alloc", 0)
        r = idx.search(xq, 20)
        idx.close()
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)
    assert failed >= 1


def test_range_and_kmeans_allocation_failures(vs):
    xb = syn.normal_unit(3000, 64, 4, 0)
    xq = np.concatenate([xb[:20] + 0.01, syn.normal_unit(20, 64, 4, 1)]).astype(np.float32)
    lims, D, I = oracle.flat_range_search(xb, xq, 0.05, 0, NT)
    idx = vs.GpuIndexFlat.l2(64, storage="f32")
    idx.add(xb)
    idx.set_option("fail_alloc", 1)
    _oom(vs, lambda: idx.range_search(xq, 0.05))
    idx.set_option("fail_alloc", 0)
    rr = idx.range_search(xq, 0.05)
    assert_range_parity(rr.limits, rr.distances, rr.ids, lims, D, I)

    cen = xb[:50].copy()
    u = syn.rng(5, 0).random(50 * 64)
    idx.set_option("fail_alloc", 1)
    _oom(vs, lambda: vs.kmeans_step(idx, cen, 1, u))
    idx.set_option("fail_alloc", 0)
    a, newc, cnt, obj = vs.kmeans_step(idx, cen, 1, u)
    idx.close()
    ar, _, objr = oracle.kmeans_assign(xb, cen, NT)
    assert np.array_equal(a, ar) and obj == objr


def test_device_probes(vs):
    """vs_dev_probe: read bandwidth (what 0), bf16 MFMA rate on small-integer
    (1) and random (2) operands, all positive and below the published peaks
    (8 TB/s, 2.5 PFLOP/s); other codes are rejected."""
    import ctypes
    from vector_store import _native as N

    lib = N.load()
    vals = {}
    for what, nbytes in ((0, 1 << 28), (1, 0), (2, 0)):
        v = ctypes.c_double(0.0)
        assert lib.vs_dev_probe(0, what, nbytes, ctypes.byref(v)) == 0
        vals[what] = v.value
    assert 500.0 < vals[0] < 8000.0
    assert 100.0 < vals[1] <= 2600.0 and 100.0 < vals[2] <= 2600.0
    v = ctypes.c_double(0.0)
    assert lib.vs_dev_probe(0, 3, 0, ctypes.byref(v)) == N.VS_ERR_INVALID


@pytest.mark.parametrize("storage", ["f32", "bf16", "auto"])
def test_add_is_all_or_nothing(vs, storage):
    """Rows are stored while they are checked: an add that meets a NaN leaves
    the index as it was, and so does the space it had written to (the next
    add, and tiles read past the last row, find zeros there)."""
    xb, xq = syn.int_grid(700, 24, 3, 0), syn.int_grid(9, 24, 3, 1)
    idx = vs.GpuIndexFlat.l2(24, storage=storage)
    idx.add(xb[:300])
    bad = xb[300:].copy()
    bad[333, 7] = np.nan
    with pytest.raises(vs.VsError):
        idx.add(bad)
    assert idx.ntotal == 300
    for rows in (xb[:300], xb):
        if len(rows) > 300:
            idx.add(xb[300:])
        idx.set_option("direct", 0)
        r = idx.search(xq, 12)
        Dr, Ir = oracle.flat_search(rows, xq, 12, 0, NT)
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=rows, xq=xq)
    if storage == "auto":  # and one that widens the storage
        idx.add(xb[:50] + np.float32(0.3))
        rows = np.concatenate([xb, xb[:50] + np.float32(0.3)])
        r = idx.search(xq, 12)
        Dr, Ir = oracle.flat_search(rows, xq, 12, 0, NT)
        assert idx.storage == "f32"
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=rows, xq=xq)
    idx.close()


def _copied(vs, xb, xq, k):
    """An index of fp32 rows that holds their copy (built by its second search)."""
    idx = vs.GpuIndexFlat.l2(xb.shape[1], storage="f32")
    idx.set_option("direct", 0)
    idx.add(xb)
    for _ in range(2):
        idx.search(xq, k)
    return idx


def test_search_gives_up_its_own_copy(vs):
    """Scratch that does not fit beside the search's own row copy: the copy
    goes, and the call succeeds without it."""
    from vector_store import _native as NN

    xb, xq = syn.normal_unit(20_000, 96, 3, 0), syn.normal_unit(200, 96, 3, 1)
    Dr, Ir = oracle.flat_search(xb, xq, 10, 0, NT)
    lims, Dx, Ix = oracle.flat_range_search(xb, xq, 1.6, 0, NT)
    qb, Db, Ib = NN.DeviceBuffer(xq.nbytes), NN.DeviceBuffer(200 * 40), NN.DeviceBuffer(200 * 40)
    qb.upload(xq)
    D, I = np.empty((200, 10), np.float32), np.empty((200, 10), np.int32)
    for n in (1, 2, 3):
        idx = _copied(vs, xb, xq[:5], 10)
        idx.set_option("fail_alloc", n)
        idx.search_device(qb, 200, 10, Db, Ib)
        idx.set_option("fail_alloc", 0)
        assert idx.prof_get("copy_given_up")[0] == 1
        Db.download(D)
        Ib.download(I)
        assert_knn_parity(D, I, Dr, Ir, 0, rtol=0.0, atol=0.0)
        r = idx.search(xq, 10)
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0)
        idx.close()
    idx = _copied(vs, xb, xq[:5], 10)
    idx.set_option("fail_alloc", 2)  # (the first is the query staging, before the rows are chosen)
    rr = idx.range_search(xq, 1.6)
    idx.set_option("fail_alloc", 0)
    assert idx.prof_get("copy_given_up")[0] == 1
    idx.close()
    for b in (qb, Db, Ib):
        b.free()
    assert_range_parity(rr.limits, rr.distances, rr.ids, lims, Dx, Ix)


@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_no_room_for_the_key_matrix(vs, storage):
    """A small search whose exact keys (its second and third allocation) do not
    fit takes the selection, which then reads host queries from pinned memory."""
    from vector_store import _native as NN

    xb, xq = syn.int_grid(5000, 64, 3, 0), syn.int_grid(6, 64, 3, 1)
    Dr, Ir = oracle.flat_search(xb, xq, 10, 0, NT)
    qb, Db, Ib = NN.DeviceBuffer(xq.nbytes), NN.DeviceBuffer(240), NN.DeviceBuffer(240)
    qb.upload(xq)
    D, I = np.empty((6, 10), np.float32), np.empty((6, 10), np.int32)
    for n in (2, 3):
        idx = vs.GpuIndexFlat.l2(64, storage=storage)
        idx.add(xb)
        idx.set_option("fail_alloc", n)  # (the first is the pinned control block)
        idx.search_device(qb, 6, 10, Db, Ib)
        assert idx.prof_get("direct")[0] == 0
        Db.download(D)
        Ib.download(I)
        assert_knn_parity(D, I, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)
        idx.search_device(qb, 6, 10, Db, Ib)
        assert idx.prof_get("direct")[0] == 1
        idx.close()
        idx = vs.GpuIndexFlat.l2(64, storage=storage)
        idx.add(xb)
        idx.set_option("fail_alloc", n)
        r = idx.search(xq, 10)
        idx.set_option("fail_alloc", 0)
        idx.close()
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)
    for b in (qb, Db, Ib):
        b.free()


def test_idle_copies_are_given_back(vs):
    """An allocation that finds the device full takes the row copies of other
    indexes and succeeds; their next searches are exact, and copy again."""
    xb, xq = syn.normal_unit(20_000, 96, 3, 0), syn.normal_unit(20, 96, 3, 1)
    Dr, Ir = oracle.flat_search(xb, xq, 10, 0, NT)
    a, c = _copied(vs, xb, xq, 10), _copied(vs, xb, xq, 10)
    b = vs.GpuIndexFlat.l2(96, storage="f32")
    b.set_option("full_alloc", 1)
    b.add(xb[:100])  # (its storage is the first allocation)
    b.set_option("full_alloc", 0)
    assert a.prof_get("copy_taken")[0] == 1 and c.prof_get("copy_taken")[0] == 1
    for idx in (a, c):
        for _ in range(3):
            r = idx.search(xq, 10)
            assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0)
    b.set_option("full_alloc", 1)
    b.reserve(5000)
    b.set_option("full_alloc", 0)
    assert a.prof_get("copy_taken")[0] == 2  # (it had copied again)
    a.close()
    c.close()
    b.set_option("full_alloc", 1)  # no copy left to take
    _oom(vs, lambda: b.reserve(50_000))
    b.set_option("full_alloc", 0)
    b.close()


def test_copies_taken_by_another_thread(vs):
    """One thread searches on row copies, changes its rows and searches again
    while another allocates on a full device: every result is exact, whether
    the copy was idle (taken) or in use (left alone)."""
    import threading

    xb, xq = syn.normal_unit(30_000, 96, 3, 0), syn.normal_unit(40, 96, 3, 1)
    Dr, Ir = oracle.flat_search(xb, xq, 10, 0, NT)
    Dh, Ih = oracle.flat_search(xb[:20_000], xq, 10, 0, NT)
    errors, done = [], threading.Event()

    def searches():
        try:
            idx = vs.GpuIndexFlat.l2(96, storage="f32")
            idx.set_option("direct", 0)
            for _ in range(6):
                idx.reset()
                for rows, D, I in ((xb[:20_000], Dh, Ih), (xb[20_000:], Dr, Ir)):
                    idx.add(rows)
                    for _ in range(4):
                        r = idx.search(xq, 10)
                        assert_knn_parity(r.distances, r.ids, D, I, 0, rtol=0.0, atol=0.0)
            idx.close()
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)
        finally:
            done.set()

    t = threading.Thread(target=searches)
    t.start()
    turns = 0
    while not done.wait(0.002) and turns < 2000:
        turns += 1
        b = vs.GpuIndexFlat.l2(96, storage="f32")
        b.set_option("full_alloc", 1)
        try:
            b.reserve(1000)
        except vs.VsError as e:  # no idle copy at that moment
            assert e.code == vs._native.VS_ERR_OOM
        b.set_option("full_alloc", 0)
        b.close()
    t.join()
    assert not errors, errors
    assert turns > 0


def test_failed_add_keeps_the_storage(vs):
    """A host add of more than one upload chunk (256 MiB) whose first rows bf16
    does not hold and whose last row is not finite: the storage stays bf16."""
    d, n = 4096, 16_500
    xb, xq = syn.int_grid(300, d, 3, 0), syn.int_grid(5, d, 3, 1)
    idx = vs.GpuIndexFlat.l2(d)
    idx.add(xb)
    bad = np.zeros((n, d), np.float32)
    bad[0, 0] = 0.3
    bad[-1, -1] = np.inf
    with pytest.raises(vs.VsError) as e:
        idx.add(bad)
    assert e.value.code == vs._native.VS_ERR_NONFINITE
    assert idx.ntotal == 300 and idx.storage == "bf16"
    idx.set_option("direct", 0)
    r = idx.search(xq, 12)
    Dr, Ir = oracle.flat_search(xb, xq, 12, 0, NT)
    assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0, xb=xb, xq=xq)
    bad[-1, -1] = 1.0  # and one that widens it
    idx.add(bad)
    assert idx.storage == "f32" and idx.ntotal == 300 + n
    assert np.array_equal(idx.reconstruct_n(299, 2), np.concatenate([xb[299:], bad[:1]]))
    assert np.array_equal(idx.reconstruct(300 + n - 1), bad[-1])
    idx.close()


def test_range_gives_its_sort_space_back(vs):
    """2e7 hits take 880 MB while they are scored and sorted; the index keeps
    the candidates' 160 MB."""
    import ctypes

    def free():
        f, t = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert vs.load().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    xb, xq = syn.normal_unit(5000, 8, 3, 0), syn.normal_unit(4000, 8, 3, 1)
    idx = vs.GpuIndexFlat.l2(8, storage="f32")
    idx.add(xb)
    idx.range_search(xq[:10], 1e9)
    before = free()
    rr = idx.range_search(xq, 1e9)
    kept = before - free()
    idx.close()
    assert rr.limits[-1] == 20_000_000
    assert kept <= 400e6, f"{kept / 1e6:.0f} MB kept"


@pytest.mark.parametrize("first", [0, 3000])
def test_widening_add_holds_its_rows_once(vs, first):
    """An add that widens automatic storage needs room for its rows in fp32, not
    beside their bf16 storage as well: 805 MB and the 268 MB of staging."""
    import ctypes
    import threading

    lib = vs.load()
    f, t = ctypes.c_size_t(0), ctypes.c_size_t(0)

    def free():
        assert lib.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    d, n = 4096, 49_152
    xb = np.zeros((n, d), np.float32)
    xb[0, 0] = xb[-1, -1] = 0.3
    head = syn.int_grid(first, d, 3, 0) if first else None
    idx = vs.GpuIndexFlat.l2(d)
    if first:
        idx.add(head)
    idx.reconstruct_n(0, first)
    before, low, done = free(), [1 << 60], threading.Event()

    def poll():
        while not done.wait(0.001):
            low[0] = min(low[0], free())

    th = threading.Thread(target=poll)
    th.start()
    idx.add(xb)
    done.set()
    th.join()
    used = before - low[0]
    assert idx.storage == "f32" and idx.ntotal == first + n
    if first:
        assert np.array_equal(idx.reconstruct_n(0, first), head)
    assert np.array_equal(idx.reconstruct_n(first, 1)[0], xb[0])
    assert np.array_equal(idx.reconstruct(first + n - 1), xb[-1])
    idx.close()
    assert used <= 1.25e9, f"{used / 1e6:.0f} MB at the most"
