"""Rows long enough that a scan's query block only just fits the LDS, or no
longer does: range search takes every dimension up to the block's own size, a
query that has to be searched again is, and a call gives the same answer
whether it is the first on its rows or a later one (on their copy)."""
import numpy as np
import pytest

import oracle
from _parity import assert_knn_parity, assert_range_parity
from vector_store import synthetic as syn

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()


def _bf16(x):
    return syn.bf16_bits_to_f32(syn.to_bf16_bits(x))


def _index(vs, xb, metric, storage, **options):
    idx = vs.GpuIndexFlat(xb.shape[1], vs.Metric(metric), storage=storage)
    idx.set_option("direct", 0)
    for name, value in options.items():
        idx.set_option(name, value)
    idx.add(xb)
    return idx


# the longest rows of the streaming scan, whose 16-query block then fills the
# LDS but for 64-entry wave buffers: two query planes beside fp32 rows and
# beside bf16 rows, and one plane
EDGES = [("f32", 2496, False), ("f32", 2400, False), ("bf16", 2432, False), ("bf16", 4992, True),
         ("f32", 4992, True)]


@pytest.mark.parametrize("storage,d,bf16_queries", EDGES)
@pytest.mark.parametrize("copy16", [0, 1])
def test_range_at_the_longest_rows(vs, storage, d, bf16_queries, copy16):
    xb, xq = syn.normal_unit(600, d, d, 0), syn.normal_unit(9, d, d, 1)
    xb[:90] = np.repeat(xq, 10, axis=0) + 0.005 * xb[:90]
    if storage == "bf16":
        xb = _bf16(xb)
    if bf16_queries:
        xq = _bf16(xq)
    for metric, radius in ((0, 0.5), (1, 0.8)):
        idx = _index(vs, xb, metric, storage, copy16=copy16)
        got = [idx.range_search(xq, radius) for _ in range(2)]
        idx.close()
        lims, D, I = oracle.flat_range_search(xb, xq, radius, metric, NT)
        assert lims[-1] >= 90
        for rr in got:
            assert_range_parity(rr.limits, rr.distances, rr.ids, lims, D, I)


@pytest.mark.parametrize("storage,d,bf16_queries", EDGES)
def test_unproven_queries_of_the_longest_rows(vs, storage, d, bf16_queries):
    """Near-copies of the queries, closer to each other than the selection's
    error: every query is searched again."""
    g = syn.rng(d, 5)
    base = syn.normal_unit(3, d, d, 6)
    xb = np.concatenate([np.repeat(base, 200, axis=0), syn.normal_unit(400, d, d, 7)])
    j = g.integers(0, d, (600, 4))
    for r in range(600):  # a few elements moved by less than the others' rounding
        xb[r, j[r]] *= np.float32(1.0 + 2.0 ** -12 if storage == "f32" else 1.0 + 2.0 ** -7)
    if storage == "bf16":
        xb = _bf16(xb)
    xq = _bf16(base) if bf16_queries else base
    for metric in (0, 1):
        idx = _index(vs, xb, metric, storage, copy16=0)
        idx.prof_reset()
        r = idx.search(xq, 10)
        again = idx.prof_get("exact_fallback")[0]
        idx.close()
        Dr, Ir = oracle.flat_search(xb, xq, 10, metric, NT)
        assert_knn_parity(r.distances, r.ids, Dr, Ir, metric, rtol=0.0, atol=0.0)
        assert storage == "bf16" or again == 3


def _close_rows(base, n, d, seed):
    """n rows per base row: it with a few elements moved by less than bf16 sees."""
    xb = np.repeat(base, n, axis=0)
    j = syn.rng(seed, 5).integers(0, d, (len(xb), 4))
    for r in range(len(xb)):
        xb[r, j[r]] *= np.float32(1.0 + 2.0 ** -12)
    return xb


@pytest.mark.parametrize("d,copy16", [(3072, 0), (6000, 1)])
def test_few_unproven_queries_of_a_large_batch(vs, d, copy16):
    """The GEMM-tiled scan takes rows of any length, from 512 queries on; the
    three queries it cannot prove have no scan of their own."""
    base = syn.normal_unit(3, d, d, 6)
    xb = np.concatenate([_close_rows(base, 100, d, d), syn.normal_unit(500, d, d, 7)])
    xq = np.concatenate([base, syn.normal_unit(517, d, d, 8)])
    for metric in (0, 1):
        idx = _index(vs, xb, metric, "f32", copy16=copy16)
        for _ in range(2):
            r = idx.search(xq, 10)
            s = np.arange(0, 520) < 20
            Dr, Ir = oracle.flat_search(xb, xq[s], 10, metric, NT)
            assert_knn_parity(r.distances[s], r.ids[s], Dr, Ir, metric, rtol=0.0, atol=0.0)
        idx.close()


def test_query_past_bf16_on_the_copy(vs):
    """Found short on the copy, then without a scan of the rows themselves."""
    d = 3072
    xb, xq = syn.normal_unit(1500, d, d, 0), syn.normal_unit(150, d, d, 1)
    xq[2] /= np.abs(xq[2]).max()
    xq[2] *= np.float32(3.4e38)
    xb *= np.float32(1e-3)
    idx = _index(vs, xb, 1, "f32")
    Dr, Ir = oracle.flat_search(xb, xq, 10, 1, NT)
    for _ in range(2):
        r = idx.search(xq, 10)
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 1, rtol=0.0, atol=0.0)
    idx.close()


# fp32 rows whose own scan does not fit (one exists on the copy up to 4,736
# elements, none at 6,000): the first call, a later one, and with the copy off
@pytest.mark.parametrize("d,nq,k", [(3072, 8, 10), (3000, 70, 25), (4990, 5, 3), (6000, 4, 10),
                                    (3072, 3, 300)])
def test_first_and_later_calls_agree(vs, d, nq, k):
    xb, xq = syn.normal_unit(1500, d, d, 0), syn.normal_unit(nq, d, d, 1)
    for copy16 in (1, 0):
        for metric in (0, 1):
            idx = _index(vs, xb, metric, "f32", copy16=copy16)
            got = [idx.search(xq, k) for _ in range(3)]
            idx.close()
            Dr, Ir = oracle.flat_search(xb, xq, k, metric, NT)
            for r in got:
                assert_knn_parity(r.distances, r.ids, Dr, Ir, metric, rtol=0.0, atol=0.0)


@pytest.mark.parametrize("d", [2600, 3072])
def test_first_range_search(vs, d):
    xb, xq = syn.normal_unit(1500, d, d, 0), syn.normal_unit(6, d, d, 1)
    xb[:30] = np.repeat(xq, 5, axis=0) + 0.005 * xb[:30]
    idx = _index(vs, xb, 0, "f32")
    got = [idx.range_search(xq, 0.5) for _ in range(2)]
    idx.close()
    lims, D, I = oracle.flat_range_search(xb, xq, 0.5, 0, NT)
    for rr in got:
        assert_range_parity(rr.limits, rr.distances, rr.ids, lims, D, I)


def test_long_rows_report_nonfinite_queries(vs):
    xb, xq = syn.normal_unit(700, 6000, 1, 0), syn.normal_unit(3, 6000, 1, 1)
    for storage, bits in (("f32", False), ("bf16", False), ("bf16", True)):
        idx = _index(vs, xb, 0, storage)
        bad = xq.copy()
        bad[1, 5] = np.nan
        with pytest.raises(vs.VsError) as e:
            idx.search(syn.to_bf16_bits(bad) if bits else bad, 4)
        assert e.value.code == vs._native.VS_ERR_NONFINITE
        rows = xb if storage == "f32" else _bf16(xb)
        q = _bf16(xq) if bits else xq
        r = idx.search(syn.to_bf16_bits(xq) if bits else xq, 4)
        idx.close()
        Dr, Ir = oracle.flat_search(rows, q, 4, 0, NT)
        assert_knn_parity(r.distances, r.ids, Dr, Ir, 0, rtol=0.0, atol=0.0)
