"""Exact top-k over sets of buckets (grab_bucket_scan_topk) against the CPU's exact label-set scan."""
import numpy as np
import pytest

import datasets

pytestmark = pytest.mark.gpu


def _case(grab, n, dim, n_buckets, nq, seed, unit, empty=()):
    """Rows stored bucket by bucket with Zipf-sized buckets (the listed ones empty), queries with 1-4 buckets each."""
    rng = np.random.default_rng(seed)
    labels = np.sort(datasets.zipf_labels(n, n_buckets, 1.1, seed + 1))
    for b in empty:
        labels[labels == b] = (b + 1) % n_buckets
    labels = np.sort(labels)
    data = datasets.unit_rows(n, dim, seed + 2) if unit else datasets.mixture(n, dim, 12, seed + 2, seed + 3)
    q = datasets.unit_rows(nq, dim, seed + 4) if unit else datasets.mixture(nq, dim, 12, seed + 2, seed + 5)
    masks = datasets.label_masks(nq, n_buckets, seed + 6)
    offsets = np.searchsorted(labels, np.arange(n_buckets + 1)).astype(np.uint64)
    return data, labels, q, masks, offsets, rng


@pytest.mark.parametrize("n,dim,n_buckets,nq,k,metric,unit", [
    (6000, 128, 8, 300, 10, 0, False),      # integer rows: ties between equal distances go to the lower id
    (20000, 64, 64, 700, 10, 1, True),      # inner product on unit rows, 64 buckets
    (50000, 32, 5, 129, 33, 0, True),       # buckets longer than one piece of 16384 columns, k above 32
    (3000, 768, 64, 64, 10, 1, True),       # the row length of the high-dimensional configuration
    (50000, 32, 5, 129, 16, 0, False),      # the longest lists that are selected from stored distances: buckets in pieces ...
    (50000, 32, 5, 129, 17, 0, False),      # ... and the shortest beyond
    (4200, 32, 64, 5000, 1, 0, False),      # more row tiles than one pass takes, a ragged last column tile
])
def test_bucket_scan_equals_the_cpu_label_scan(oracle, grab, n, dim, n_buckets, nq, k, metric, unit):
    data, labels, q, masks, offsets, _ = _case(grab, n, dim, n_buckets, nq, 7 * n_buckets + dim, unit)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ids, dist, _ = grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, nq, k, masks, metric=metric)
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=metric, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks)
    bad = np.flatnonzero((ids != eids).any(axis=1))
    assert bad.size == 0, f"queries {bad[:5]}: {ids[bad[0]]} vs {eids[bad[0]]}"
    assert np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
    # and the GPU's own scan of every row with the label test
    gids, gdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, metric=metric, filter_kind=grab.FILTER_MASK,
                                          d_labels=grab.DeviceArray.from_numpy(labels), d_masks=grab.DeviceArray.from_numpy(masks))
    assert np.array_equal(ids, gids) and np.array_equal(dist.view(np.uint32), gdist.view(np.uint32))


def test_bucket_scan_queries_that_the_candidates_cannot_prove(oracle, grab):
    # rows that all sit within 0.01 of each other far from the origin: the distances between them are far below the
    # rounding error of |a|^2 + |b|^2 - 2ab, a merged candidate list proves nothing, and every query takes the plain way
    # (a problem per tile-grid row, whose own check sends it on to the scan of every admissible column)
    n, dim, nb, nq, k = 5000, 64, 6, 150, 10
    rng = np.random.default_rng(4)
    data = (np.float32(1000.0) + np.float32(0.01) * rng.standard_normal((n, dim))).astype(np.float32)
    q = (np.float32(1000.0) + np.float32(0.01) * rng.standard_normal((nq, dim))).astype(np.float32)
    labels = np.sort(rng.integers(0, nb, n)).astype(np.uint8)
    masks = datasets.label_masks(nq, nb, 8)
    offsets = np.searchsorted(labels, np.arange(nb + 1)).astype(np.uint64)
    ids, dist, _ = grab.bucket_scan_topk(grab.DeviceArray.from_numpy(data), n, dim, offsets, grab.DeviceArray.from_numpy(q), nq, k, masks)
    sent_on = grab.last_knn_exact_rows()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
    assert sent_on > nq // 2, sent_on


def test_bucket_scan_leaves_out_what_has_no_order(oracle, grab):
    # columns whose |a|^2 + |b|^2 - 2ab is no number are no candidates, in buckets below and above 512 rows, whichever way
    # the list is selected (stored distances up to k = 16, inside the contraction beyond)
    n, dim = 4000, 32
    offsets = np.array([0, 300, 1500, 4000], np.uint64)
    data, q = datasets.mixture(n, dim, 12, 1, 2), datasets.mixture(4, dim, 12, 1, 3)
    data[320:900:7, 5] = 0.0  # against an infinite query 0 * inf, beside distances that are infinite
    q[1, 3], q[2, 5] = np.nan, -np.inf
    bad = data.copy()
    bad[100:700] = np.nan
    bad[2000] = -np.float32(np.nan)
    for rows, gone in ((data, []), (bad, [*range(100, 700), 2000])):
        d_rows, d_q = grab.DeviceArray.from_numpy(rows), grab.DeviceArray.from_numpy(q)
        for mask in (1, 2, 4, 7):
            masks = np.full(4, mask, np.uint64)
            long_ids, long_dist, _ = grab.bucket_scan_topk(d_rows, n, dim, offsets, d_q, 4, 17, masks)
            labels = np.repeat(np.arange(3), np.diff(offsets.astype(np.int64))).astype(np.uint8)
            labels[gone] = 63
            eids, edist = oracle.bruteforce_topk(data, q[[0, 3]], 16, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks[:2])
            for k in (10, 16):
                ids, dist, _ = grab.bucket_scan_topk(d_rows, n, dim, offsets, d_q, 4, k, masks)
                assert np.array_equal(ids, long_ids[:, :k]) and np.array_equal(dist.view(np.uint32), long_dist[:, :k].view(np.uint32)), (mask, k)
                assert (ids[1] == -1).all()
                assert np.array_equal(ids[[0, 3]], eids[:, :k]) and np.array_equal(dist[[0, 3]], edist[:, :k]), (mask, k)


def test_bucket_scan_short_and_empty_buckets(oracle, grab):
    # buckets with fewer rows than k, empty buckets, queries whose buckets are all empty, a mask bit beyond the buckets
    n, dim, nb, nq, k = 900, 32, 16, 200, 20
    data, labels, q, masks, offsets, rng = _case(grab, n, dim, nb, nq, 3, False, empty=(2, 9, 15))
    masks[:5] = np.uint64(1 << 2)                       # only an empty bucket
    masks[5:9] = np.uint64((1 << 9) | (1 << 15))
    masks[9] = np.uint64((1 << 40) | (1 << 3))          # a bucket that does not exist is ignored
    sizes = np.diff(offsets.astype(np.int64))
    assert (sizes == 0).sum() >= 3 and ((sizes > 0) & (sizes < k)).any()
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ids, dist, _ = grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, nq, k, masks)
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_MASK, labels=labels,
                                         masks=masks & np.uint64((1 << nb) - 1))
    assert np.array_equal(ids, eids)
    assert (ids[:9] == -1).all() and (ids[9] >= 0).any()
    valid = ids >= 0
    assert np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])
    # all queries empty
    ids0, _, _ = grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, 4, k, masks[:4])
    assert (ids0 == -1).all()
    # argument errors
    import ctypes as C
    bad = offsets.copy()
    bad[3] = bad[4] + 1
    assert grab.lib.grab_bucket_scan_topk(C.c_void_p(d_data.ptr), C.c_size_t(n), C.c_uint32(dim), bad.ctypes.data_as(C.c_void_p),
                                          C.c_uint32(nb), C.c_void_p(d_q.ptr), C.c_size_t(4), C.c_uint32(k), C.c_int(0),
                                          masks.ctypes.data_as(C.c_void_p), C.c_void_p(d_data.ptr), C.c_void_p(d_data.ptr), None, None) == 1
    assert b"offsets" in grab.lib.grab_last_error()


@pytest.mark.parametrize("n,dim,nb,nq,k,metric,per_query", [(30000, 64, 64, 400, 10, 0, 64), (40000, 96, 7, 1200, 128, 1, 3), (5000, 32, 64, 900, 20, 0, 9)])
def test_bucket_scan_on_f16_rows_with_many_buckets_a_query(oracle, grab, n, dim, nb, nq, k, metric, per_query):
    # the lists of all of a query's buckets are put together under one threshold: all 64 of them, few large ones, many small ones
    rng = np.random.default_rng(n)
    data = datasets.unit_rows(n, dim, 3) if metric else datasets.mixture(n, dim, 12, 3, 4)
    q = datasets.unit_rows(nq, dim, 5) if metric else datasets.mixture(nq, dim, 12, 3, 6)
    labels = np.sort(datasets.zipf_labels(n, nb, 1.1, 5))
    offsets = np.searchsorted(labels, np.arange(nb + 1)).astype(np.uint64)
    masks = np.array([np.bitwise_or.reduce(np.uint64(1) << rng.choice(nb, per_query, replace=False).astype(np.uint64)) for _ in range(nq)], np.uint64)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ids, dist, _ = grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, nq, k, masks, metric=metric)
    assert grab.last_knn_f16_flop() > 0
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=metric, filter_kind=oracle.FILTER_MASK, labels=labels.astype(np.uint8), masks=masks)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


@pytest.mark.parametrize("k", [10, 128])
def test_bucket_scan_of_large_buckets(oracle, grab, k):
    # a query's sixty pieces list 900 columns give or take 600: as many as a wave scores, as it holds, and more, of which it takes
    # the nearest
    n, dim, nq = 1_000_000, 32, 300
    data, q = datasets.gaussian(n, dim, 4), datasets.gaussian(nq, dim, 7)
    offsets = np.array([0, 400_000, 400_050, 950_000, n], np.uint64)
    masks = np.where(np.arange(nq) % 2, np.uint64(5), np.uint64(7)).astype(np.uint64)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, n, dim, 0)
    ids, dist, _ = base.bucket_topk(offsets, d_q, nq, k, masks)
    assert grab.last_knn_f16_flop() > 0
    if k == 10:
        assert grab.last_knn_stats()[1] <= 5
    base.close()
    labels = np.repeat(np.arange(4, dtype=np.uint8), np.diff(offsets.astype(np.int64)))
    gids, gdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, filter_kind=grab.FILTER_MASK, d_labels=grab.DeviceArray.from_numpy(labels),
                                          d_masks=grab.DeviceArray.from_numpy(masks))
    assert np.array_equal(ids, gids) and np.array_equal(dist.view(np.uint32), gdist.view(np.uint32))
    eids, _ = oracle.bruteforce_topk(data, q[:8], k, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks[:8])
    assert np.array_equal(ids[:8], eids)
