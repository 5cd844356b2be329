"""Searches on the exact key matrix (small searches, and k beyond the fused
selection's lists) against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle
from _parity import assert_knn_parity
from vector_store import synthetic as syn

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()


def _check(vs, xb, xq, k, metric, storage, **options):
    idx = vs.GpuIndexFlat(xb.shape[1], vs.Metric(metric), storage=storage)
    for name, value in options.items():
        idx.set_option(name, value)
    idx.add(xb)
    r = idx.search(xq, k)
    n = idx.prof_get("direct")[0]
    idx.close()
    Dr, Ir = oracle.flat_search(xb, xq, k, metric, NT)
    assert_knn_parity(r.distances, r.ids, Dr, Ir, metric, rtol=0.0, atol=0.0)
    return n


# tile edges: 64 rows, 64-element chunks, 4 queries (one per wave) or 16
@pytest.mark.parametrize("n,d,nq,k", [(1, 1, 1, 1), (63, 3, 1, 5), (64, 64, 4, 64), (65, 65, 5, 80),
                                      (1000, 130, 16, 10), (2049, 100, 17, 2), (5000, 33, 33, 409)])
@pytest.mark.parametrize("metric,storage", [(0, "f32"), (1, "f32"), (0, "bf16"), (1, "bf16")])
def test_direct_search_edges(vs, n, d, nq, k, metric, storage):
    g = syn.rng(n + d, 3)
    xb = g.standard_normal((n, d)).astype(np.float32)
    xq = g.standard_normal((nq, d)).astype(np.float32)
    if storage == "bf16":
        xb = syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
    assert _check(vs, xb, xq, k, metric, storage) == 1


# the buffer's edges (cap = 2048 keys up to k = 1024, then the next power of
# two of 2 k), segments (n >= 65,536 and few queries), the largest k, the sort
# beyond it; ties in hundreds (integers) and one far outlier, which leaves
# the first histogram's other keys in one bin
@pytest.mark.parametrize("n,nq,k,data", [(2048, 2, 1024, "normal"), (4097, 3, 1025, "ties"),
                                         (70_000, 1, 500, "normal"), (140_000, 3, 2000, "ties"),
                                         (140_000, 40, 1000, "outlier"), (9000, 2, 8192, "normal"),
                                         (9000, 2, 8193, "normal"), (3000, 2, 5000, "ties")])
def test_key_selection(vs, n, nq, k, data):
    g = syn.rng(n, k)
    if data == "ties":
        xb = g.integers(0, 3, (n, 12)).astype(np.float32)
        xq = g.integers(0, 3, (nq, 12)).astype(np.float32)
    else:
        xb = g.standard_normal((n, 12)).astype(np.float32)
        xq = g.standard_normal((nq, 12)).astype(np.float32)
        if data == "outlier":
            xb[7] *= 1e15
    for metric in (0, 1):
        n_direct = _check(vs, xb, xq, k, metric, "f32", direct=1)
        assert n_direct == (1 if k <= 8192 else 0)


def test_direct_reports_nonfinite_queries(vs):
    """The call fails, and device results of fp32 queries on fp32 rows stay
    as they were."""
    from vector_store import _native as NN

    xb = syn.normal_unit(500, 16, 1, 0)
    xq = syn.normal_unit(6, 16, 1, 1)
    xq[4, 3] = np.nan
    idx = vs.GpuIndexFlat.ip(16, storage="f32")
    idx.add(xb)
    with pytest.raises(vs.VsError) as e:
        idx.search(xq, 3)
    assert e.value.code == NN.VS_ERR_NONFINITE
    D = np.full((6, 3), 7.0, np.float32)
    qb, Db, Ib = NN.DeviceBuffer(xq.nbytes), NN.DeviceBuffer(D.nbytes), NN.DeviceBuffer(D.nbytes)
    qb.upload(xq)
    Db.upload(D)
    with pytest.raises(vs.VsError):
        idx.search_device(qb, 6, 3, Db, Ib)
    out = np.empty_like(D)
    Db.download(out)
    for b in (qb, Db, Ib):
        b.free()
    xq[4, 3] = 0.5
    r = idx.search(xq, 3)
    idx.close()
    assert np.array_equal(out, D)
    Dr, Ir = oracle.flat_search(xb, xq, 3, 1, NT)
    assert_knn_parity(r.distances, r.ids, Dr, Ir, 1, rtol=0.0, atol=0.0)


@pytest.mark.parametrize("k", [5, 8193])
@pytest.mark.parametrize("metric", [0, 1])
def test_scores_past_fp32(vs, metric, k):
    """Rows whose score is infinite in fp32 are rows all the same (the
    reference compares the fp64 score): last or first of all 40, never a
    sentinel."""
    xb = syn.normal_unit(40, 8, 5, 0)
    xb[3] *= np.float32(3e38)
    xb[9] *= np.float32(-3e38)
    xq = (syn.normal_unit(3, 8, 5, 1) * np.float32(100.0)).astype(np.float32)
    _check(vs, xb, xq, 40 if k == 5 else k, metric, "f32")
    _check(vs, xb, xq, k, metric, "f32")


@pytest.mark.parametrize("storage,metric,d", [("f32", 0, 70), ("f32", 1, 32), ("bf16", 0, 33), ("bf16", 1, 128)])
@pytest.mark.parametrize("nq,nseg,k", [(3, 1, 5), (40, 30, 10), (5, 4, 1500), (2, 3, 8192)])
def test_subset_keys(vs, storage, metric, d, nq, nseg, k):
    """Segments of every length from 0 to past four waves' rows, pairs walked
    in index order and by segment (1,024 pairs and more), k past the subset."""
    g = syn.rng(nq, nseg)
    xb = g.standard_normal((5000, d)).astype(np.float32)
    xq = g.standard_normal((nq, d)).astype(np.float32)
    if storage == "bf16":
        xb = syn.bf16_bits_to_f32(syn.to_bf16_bits(xb))
    idx = vs.GpuIndexFlat(d, vs.Metric(metric), storage=storage)
    idx.add(xb)
    ids = g.permutation(5000).astype(np.int32)
    cut = np.sort(g.choice(5001, size=nseg * 2, replace=False))
    off = np.stack([cut[0::2]] * nq)
    ln = np.stack([(cut[1::2] - cut[0::2]) * (np.arange(nseg) % 3 != 1)] * nq)
    ln[0] = 0
    r = idx.search_subsets(xq, k, ids, off, ln)
    idx.close()
    for q in range(nq):
        rows = np.concatenate([ids[o:o + l] for o, l in zip(off[q], ln[q])]).astype(np.int64)
        m = min(k, len(rows))
        assert np.all(r.ids[q, m:] == -1)
        if m:
            order = np.sort(rows)
            Dr, Ir = oracle.flat_search(xb[order], xq[q:q + 1], m, metric, 1)
            assert np.array_equal(r.distances[q, :m], Dr[0])
            assert_knn_parity(r.distances[q:q + 1, :m], r.ids[q:q + 1, :m], Dr,
                              order[Ir].astype(np.int32), metric, rtol=0.0, atol=0.0)


def test_subset_repeats_and_bad_ids(vs):
    """A row named thousands of times (past the selection's buffer) comes back
    as often; an id outside the index fails the call."""
    xb = syn.normal_unit(100, 16, 3, 0)
    idx = vs.GpuIndexFlat.l2(16, storage="f32")
    idx.add(xb)
    ids = np.concatenate([np.full(9000, 7), np.arange(100)]).astype(np.int32)
    r = idx.search_subsets(xb[7:8] + np.float32(0.01), 20, ids, [[0]], [[len(ids)]])
    assert np.all(r.ids == 7) and np.all(r.distances == r.distances[0, 0])
    r = idx.search_subsets(xb[50:51], 20, ids, [[0]], [[len(ids)]])
    assert r.ids[0, 0] == 50
    ids[-1] = 100
    with pytest.raises(ValueError):
        idx.search_subsets(xb[:1], 2, ids, [[0]], [[len(ids)]])
    idx.close()
