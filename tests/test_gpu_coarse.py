"""One-pass selection of fp32 rows (their bf16 roundings, one MFMA pass) and
the bounded re-search of what its merge cannot prove: results equal the
oracle's bit for bit whatever the data."""
import numpy as np
import pytest

import oracle
from _parity import assert_knn_parity
from vector_store import synthetic as syn

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()


def _index(vs, xb, metric, **options):
    idx = vs.GpuIndexFlat(xb.shape[1], vs.Metric(metric), storage="f32")
    idx.set_option("direct", 0)
    for name, value in options.items():
        idx.set_option(name, value)
    idx.add(xb)
    return idx


def _check(idx, xb, xq, k, metric, sub=1):
    first = idx.search(xq, k)  # (a small batch copies the rows from its second call on)
    r = idx.search(xq, k)
    assert np.array_equal(first.distances, r.distances) and np.array_equal(first.ids, r.ids)
    s = np.arange(0, len(xq), sub)
    Dr, Ir = oracle.flat_search(xb, xq[s], k, metric, NT)
    assert_knn_parity(r.distances[s], r.ids[s], Dr, Ir, metric, rtol=0.0, atol=0.0)


# streaming, row-shared and GEMM-tiled scans; with and without an estimate
# (16,384 rows, 16 queries and up); k at the keep's edges (200: the largest)
@pytest.mark.parametrize("n,d,nq,k", [(300, 7, 3, 5), (16_383, 100, 40, 16), (16_384, 64, 16, 17),
                                      (40_000, 128, 300, 100), (30_000, 300, 600, 10),
                                      (70_000, 520, 100, 200), (270_000, 40, 257, 1),
                                      (5000, 128, 520, 201)])
@pytest.mark.parametrize("metric", [0, 1])
def test_coarse_search(vs, n, d, nq, k, metric):
    xb, xq = syn.normal_unit(n, d, n, 0), syn.normal_unit(nq, d, n, 1)
    idx = _index(vs, xb, metric)
    _check(idx, xb, xq, k, metric, sub=max(1, nq // 40))
    idx.close()


@pytest.mark.parametrize("n,d,nq,k,storage", [(20_000, 64, 20, 10, "f32"), (60_000, 128, 300, 50, "f32"),
                                              (60_000, 256, 600, 10, "f32"), (60_000, 96, 300, 10, "bf16")])
def test_tight_clusters_are_searched_again(vs, n, d, nq, k, storage):
    """Clusters tighter than the rounding: most queries need the bounded
    re-search (on bf16 rows, whose error is the accumulation's, clusters of
    near-copies do)."""
    g = syn.rng(n, 3)
    cen = g.standard_normal((40, d)).astype(np.float32)
    sigma = np.float32(0.05 if storage == "f32" else 2e-4)
    xb = (cen[g.integers(0, 40, n)] + sigma * g.standard_normal((n, d))).astype(np.float32)
    xq = (cen[g.integers(0, 40, nq)] + sigma * g.standard_normal((nq, d))).astype(np.float32)
    if storage == "bf16":
        xb = syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
        xq = syn.bf16_bits_to_f32(syn.to_bf16_bits(xq))
    for metric in (0, 1):
        idx = vs.GpuIndexFlat(d, vs.Metric(metric), storage=storage)
        idx.set_option("direct", 0)
        idx.add(xb)
        idx.prof_reset()
        _check(idx, xb, xq, k, metric, sub=max(1, nq // 30))
        again = idx.prof_get("exact_fallback")[0]
        idx.close()
        assert storage == "bf16" or metric == 1 or again > nq // 2


def test_copy_follows_the_rows(vs):
    """The bf16 copy after adds (appended, and past the capacity), removals
    (rows move, fewer remain) and a reset."""
    x = syn.normal_unit(9000, 72, 3, 0)
    xq = syn.normal_unit(30, 72, 3, 1)
    idx = _index(vs, x[:1000], 0)
    _check(idx, x[:1000], xq, 5, 0)
    idx.add(x[1000:1020])
    _check(idx, x[:1020], xq, 5, 0)
    idx.add(x[1020:])
    _check(idx, x, xq, 5, 0)
    gone = np.arange(0, 9000, 3)
    idx.remove_ids(gone)
    left = np.delete(x, gone, axis=0)
    _check(idx, left, xq, 5, 0)
    idx.reset()
    idx.add(x[5000:5100])
    _check(idx, x[5000:5100], xq, 120, 0)
    rr = idx.range_search(xq, 1.8)
    lims, D, I = oracle.flat_range_search(x[5000:5100], xq, 1.8, 0, NT)
    idx.close()
    assert np.array_equal(rr.limits, lims) and np.array_equal(rr.ids, I)


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("scale", [1e-25, 1e15, 3.395e38, 3.4e38])
def test_extreme_magnitudes(vs, scale, metric):
    """Rows whose rounding residual underflows, is large, has a square past
    fp32 (the rows are then not copied) or is itself infinite (the largest
    elements round past bf16's range): proven or searched again, never wrong."""
    xb = (syn.normal_unit(3000, 16, 4, 0)).astype(np.float32)
    xb /= np.abs(xb).max()
    xb = (xb * np.float32(scale)).astype(np.float32)
    xq = syn.normal_unit(20, 16, 4, 1) * np.float32(1e-3)
    idx = _index(vs, xb, metric)
    _check(idx, xb, xq, 7, metric)
    idx.close()


@pytest.mark.parametrize("spread", [1e12, 1e14])
def test_accumulators_past_fp32(vs, spread):
    """Operands that bf16 holds whose partial sums leave fp32's range on the
    way to a score within it: the best rows' accumulators are not numbers."""
    g = syn.rng(9, 0)
    xb = np.zeros((4000, 24), np.float32)
    xb[:, 0] = np.float32(spread) * g.random(4000, dtype=np.float32)
    xb[100:120, 0] = 1e15
    xb[100:120, 1] = -1e15 * (0.7 + 0.01 * np.arange(20))
    xq = np.zeros((20, 24), np.float32)
    xq[:, :2] = 1e24
    xq[:, 2:] = g.standard_normal((20, 22))
    for storage in ("f32", "bf16"):
        rows = xb if storage == "f32" else syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
        idx = vs.GpuIndexFlat(24, vs.Metric(1), storage=storage)
        idx.set_option("direct", 0)
        idx.add(rows)
        for _ in range(2):
            r = idx.search(xq, 9)
            Dr, Ir = oracle.flat_search(rows, xq, 9, 1, NT)
            assert_knn_parity(r.distances, r.ids, Dr, Ir, 1, rtol=0.0, atol=0.0)
        idx.close()


# streaming scan without and with an estimate, row-shared and GEMM-tiled scan
@pytest.mark.parametrize("n,d,nq", [(3000, 16, 3), (20_000, 40, 40), (20_000, 128, 300), (5000, 300, 600)])
@pytest.mark.parametrize("metric,storage", [(0, "f32"), (1, "f32"), (1, "bf16")])
def test_queries_past_bf16(vs, n, d, nq, metric, storage):
    """Queries that bf16 rounds to infinity: accumulators are not numbers, and
    the scans find fewer candidates than rows, or none."""
    xb = syn.normal_unit(n, d, 4, 0)
    xq = syn.normal_unit(nq, d, 4, 1)
    xq[:nq // 2 + 1] /= np.abs(xq[:nq // 2 + 1]).max(axis=1, keepdims=True)
    xq[:nq // 2 + 1] *= np.float32(3.4e38)
    xb *= np.float32(0.1)
    if storage == "bf16":
        xb = syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
    idx = vs.GpuIndexFlat(d, vs.Metric(metric), storage=storage)
    idx.set_option("direct", 0)
    idx.add(xb)
    for _ in range(2):
        r = idx.search(xq, 7)
        assert np.all(r.ids >= 0)
        Dr, Ir = oracle.flat_search(xb, xq[::7], 7, metric, NT)
        assert_knn_parity(r.distances[::7], r.ids[::7], Dr, Ir, metric, rtol=0.0, atol=0.0)
    idx.close()


def test_adversarial_rounding(vs):
    """Every element halfway between two bf16 values, the largest residual a
    row can have, all in one direction for half of the rows: the selection's
    order is wrong by that much, the answer is not."""
    n, d = 20_000, 128
    g = syn.rng(8, 0)
    base = 1.0 + g.integers(0, 2, (n, d)) / 128.0  # neighbours of 1 in bf16
    half = np.where(g.random((n, 1)) < 0.5, 1.0, -1.0) * (0.999 / 256.0)
    xb = (base + half).astype(np.float32)
    xq = (1.0 + g.integers(0, 2, (40, d)) / 128.0 + 0.9 / 256.0).astype(np.float32)
    for metric in (0, 1):
        idx = _index(vs, xb, metric)
        _check(idx, xb, xq, 10, metric)
        idx.close()


def test_nonfinite_queries_leave_results(vs):
    from vector_store import _native as NN

    xb, xq = syn.normal_unit(20_000, 64, 1, 0), syn.normal_unit(30, 64, 1, 1)
    xq[17, 5] = np.inf
    idx = _index(vs, xb, 0)
    D = np.full((30, 4), 7.0, np.float32)
    qb, Db, Ib = NN.DeviceBuffer(xq.nbytes), NN.DeviceBuffer(D.nbytes), NN.DeviceBuffer(D.nbytes)
    qb.upload(xq)
    Db.upload(D)
    with pytest.raises(vs.VsError) as e:
        idx.search_device(qb, 30, 4, Db, Ib)
    out = np.empty_like(D)
    Db.download(out)
    for b in (qb, Db, Ib):
        b.free()
    assert e.value.code == NN.VS_ERR_NONFINITE and np.array_equal(out, D)
    xq[17, 5] = 0.1
    _check(idx, xb, xq, 4, 0)
    idx.close()


# the pair buffers of the streaming range scan: a tile with more hits than
# they hold, and hits that fill them over many tiles
@pytest.mark.parametrize("nq,radius", [(3, 1e9), (64, 2.0), (130, 1.9)])
def test_range_hit_buffers(vs, nq, radius):
    xb, xq = syn.normal_unit(3000, 48, 6, 0), syn.normal_unit(nq, 48, 6, 1)
    for storage in ("f32", "bf16"):
        rows = xb if storage == "f32" else syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
        idx = vs.GpuIndexFlat(48, vs.Metric(0), storage=storage)
        idx.add(rows)
        rr = idx.range_search(xq, radius)
        idx.close()
        lims, D, I = oracle.flat_range_search(rows, xq, radius, 0, NT)
        assert np.array_equal(rr.limits, lims) and np.array_equal(rr.ids, I)
        assert np.array_equal(rr.distances, D)


# streaming, row-shared and GEMM-tiled scans, the smallest sample and larger ones
@pytest.mark.parametrize("n,d,nq,k", [(20_000, 384, 600, 10), (17_000, 768, 100, 10), (40_000, 64, 32, 10),
                                      (30_000, 128, 300, 30), (60_000, 256, 520, 100)])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_estimates_on_sorted_rows(vs, n, d, nq, k, storage):
    """Rows grouped by topic, and queries about the first topics: the sample
    behind the thresholds is spread over the rows, so no query is misled by it
    and searched again with full lists."""
    g = syn.rng(n, 4)
    cen = g.standard_normal((n // 50, d)).astype(np.float32)
    xb = (np.repeat(cen, 50, axis=0)[:n] + np.float32(0.3) * g.standard_normal((n, d))).astype(np.float32)
    xq = (xb[:nq] + np.float32(0.01) * g.standard_normal((nq, d))).astype(np.float32)
    if storage == "bf16":
        xb, xq = (syn.bf16_bits_to_f32(syn.to_bf16_bits(a)) for a in (xb, xq))
    idx = vs.GpuIndexFlat.l2(d, storage=storage)
    idx.set_option("direct", 0)
    idx.add(xb)
    for _ in range(2):
        idx.prof_reset()
        r = idx.search(xq, k)
        assert idx.prof_get("guess_scans")[0] == 1 and idx.prof_get("fallback")[0] <= nq // 50
    idx.close()
    Dr, Ir = oracle.flat_search(xb, xq[::9], k, 0, NT)
    assert_knn_parity(r.distances[::9], r.ids[::9], Dr, Ir, 0, rtol=0.0, atol=0.0)
