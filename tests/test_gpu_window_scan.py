"""Exact top-k inside intervals of row ids (grab_window_scan_topk) against the CPU's exact range-filtered scan."""
import ctypes as C
import time

import numpy as np
import pytest

import datasets

pytestmark = pytest.mark.gpu


def _intervals(n, nq, width_lo, width_hi, seed):
    rng = np.random.default_rng(seed)
    w = rng.integers(width_lo, width_hi + 1, nq)
    lo = rng.integers(0, np.maximum(n - w, 1))
    return lo.astype(np.uint64), np.minimum(lo + w, n).astype(np.uint64)


@pytest.mark.parametrize("n,dim,nq,k,metric,kind,widths", [
    (6000, 128, 300, 10, 0, "mix", (40, 900)),       # integer rows: ties between equal distances go to the lower id
    (40000, 64, 1500, 10, 1, "unit", (300, 500)),    # inner product, more than 1024 queries: rows as bf16 halves
    (70000, 32, 1100, 33, 0, "unit", (5, 30000)),    # intervals from shorter than k to long ones, k above 32
    (9000, 768, 130, 10, 1, "unit", (100, 2000)),    # long rows
    (30000, 132, 1200, 10, 0, "gauss", (200, 4000)), # a row length that is no whole number of 32-dimension chunks: fp32 instructions
])
def test_window_scan_equals_the_cpu_range_scan(oracle, grab, n, dim, nq, k, metric, kind, widths):
    data = {"mix": lambda: datasets.mixture(n, dim, 12, 3, 4), "unit": lambda: datasets.unit_rows(n, dim, 5),
            "gauss": lambda: datasets.gaussian(n, dim, 6)}[kind]()
    q = {"mix": lambda: datasets.mixture(nq, dim, 12, 3, 7), "unit": lambda: datasets.unit_rows(nq, dim, 8),
         "gauss": lambda: datasets.gaussian(nq, dim, 9)}[kind]()
    lo, hi = _intervals(n, nq, widths[0], widths[1], n + dim)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ids, dist, _ = grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi, metric=metric)
    ts = np.arange(n, dtype=np.uint64)
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=metric, filter_kind=oracle.FILTER_RANGE, ts=ts, win_start=lo, win_end=hi)
    bad = np.flatnonzero((ids != eids).any(axis=1))
    assert bad.size == 0, f"queries {bad[:5]}: {ids[bad[0]]} vs {eids[bad[0]]} in [{lo[bad[0]]}, {hi[bad[0]]})"
    valid = ids >= 0
    assert np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])
    assert ((ids >= lo[:, None].astype(np.int64)) & (ids < hi[:, None].astype(np.int64)))[valid].all()
    on_bf16 = dim % 32 == 0 and nq >= 1024 - 127 and n >= 4096
    assert (grab.last_knn_bf16_flop() > 0) == on_bf16
    # and the GPU's own scan of every row with the window test
    gids, gdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, metric=metric, filter_kind=grab.FILTER_RANGE,
                                          d_ts=grab.DeviceArray.from_numpy(ts), d_win_start=grab.DeviceArray.from_numpy(lo),
                                          d_win_end=grab.DeviceArray.from_numpy(hi))
    assert np.array_equal(ids, gids) and np.array_equal(dist.view(np.uint32)[valid], gdist.view(np.uint32)[valid])


def test_window_scan_empty_short_and_overlong_intervals(oracle, grab):
    n, dim, nq, k = 3000, 32, 140, 12
    data, q = datasets.mixture(n, dim, 6, 1, 2), datasets.mixture(nq, dim, 6, 1, 3)
    lo, hi = _intervals(n, nq, 1, 400, 11)
    lo[:6], hi[:6] = [5, 700, 2999, 3000, 4000, 10], [5, 600, 3000, 3000, 5000, 9]      # empty, reversed, last row, beyond the end
    lo[6], hi[6] = 2990, 1 << 40                                                       # an end far beyond the rows is cut
    lo[7], hi[7] = 0, n                                                                # every row
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ids, dist, _ = grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi)
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo,
                                         win_end=np.minimum(hi, np.uint64(n)))
    assert np.array_equal(ids, eids)
    assert (ids[[0, 1, 3, 4, 5]] == -1).all() and ids[2, 0] == 2999 and (ids[2, 1:] == -1).all()
    assert (ids[6] >= 0).sum() == 10 and (ids[7] >= 0).all()
    valid = ids >= 0
    assert np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])
    # no query admits a row
    ids0, _, _ = grab.window_scan_topk(d_data, n, dim, d_q, 3, k, np.array([4, 9, 3000], np.uint64), np.array([4, 2, 3000], np.uint64))
    assert (ids0 == -1).all()
    with pytest.raises(grab.GrabError):
        grab.window_scan_topk(d_data, n, dim, d_q, nq, 200, lo, hi)


def test_window_scan_queries_that_the_candidates_cannot_prove(oracle, grab):
    # rows within 0.01 of each other far from the origin: a candidate list of GEMM-form keys proves nothing there, and
    # the queries take the plain way (a problem per query row, whose own check goes on to the scan of the interval)
    n, dim, nq, k = 5000, 64, 150, 10
    rng = np.random.default_rng(4)
    data = (np.float32(1000.0) + np.float32(0.01) * rng.standard_normal((n, dim))).astype(np.float32)
    q = (np.float32(1000.0) + np.float32(0.01) * rng.standard_normal((nq, dim))).astype(np.float32)
    lo, hi = _intervals(n, nq, 100, 1500, 12)
    ids, dist, _ = grab.window_scan_topk(grab.DeviceArray.from_numpy(data), n, dim, grab.DeviceArray.from_numpy(q), nq, k, lo, hi)
    sent_on = grab.last_knn_exact_rows()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
    assert sent_on > nq // 2, sent_on


def test_prepared_base_gives_the_same_answers_call_after_call(oracle, grab):
    # the base's rows are split once and the calls' scratch is kept: a large call, a small one, another metric's base,
    # the bucket scan on the same base - every answer equal to the one-shot entry points'
    n, dim, k = 30000, 64, 10
    data = datasets.unit_rows(n, dim, 31)
    d_data = grab.DeviceArray.from_numpy(data)
    free0 = grab.device_memory()[0]
    for metric in (0, 1):
        base = grab.ScanBase(d_data, n, dim, metric)
        for nq, widths, seed in ((1500, (200, 3000), 1), (70, (10, 400), 2), (1500, (50, 9000), 3)):
            q = datasets.unit_rows(nq, dim, 40 + seed)
            d_q = grab.DeviceArray.from_numpy(q)
            lo, hi = _intervals(n, nq, widths[0], widths[1], seed)
            ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
            assert grab.last_knn_bf16_flop() > 0      # the base holds split rows, so small calls use them too
            eids, edist, _ = grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi, metric=metric)
            assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
            oids, _ = oracle.bruteforce_topk(data, q[:40], k, metric=metric, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64),
                                             win_start=lo[:40], win_end=hi[:40])
            assert np.array_equal(ids[:40], oids)
        labels = np.sort(datasets.zipf_labels(n, 16, 1.1, 5))
        offsets = np.searchsorted(labels, np.arange(17)).astype(np.uint64)
        masks = datasets.label_masks(300, 16, 6)
        d_q = grab.DeviceArray.from_numpy(datasets.unit_rows(300, dim, 50))
        ids, dist, _ = base.bucket_topk(offsets, d_q, 300, k, masks)
        eids, edist, _ = grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, 300, k, masks, metric=metric)
        assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
        base.close()
    assert grab.device_memory()[0] >= free0 - (8 << 20)   # a closed base gives its memory back


def test_index_handle_scans_windows_exactly(oracle, grab):
    # the handle's exact range search: rows in timestamp order (several rows per timestamp) go through the prepared
    # base, which is remade after an insert; rows in any other order are scanned with the window test
    n0, n1, dim, k, nq = 6000, 1500, 64, 10, 300
    data = datasets.mixture(n0 + n1, dim, 20, 3, 4)
    ts = (np.arange(n0 + n1, dtype=np.uint64) // 7) * 3
    q = datasets.mixture(nq, dim, 20, 3, 5)
    rng = np.random.default_rng(6)
    ws = rng.integers(0, int(ts[n0 - 1]), nq).astype(np.uint64)
    we = ws + rng.integers(1, 600, nq).astype(np.uint64)
    ws[:3], we[:3] = [10**9, 50, 0], [10**9 + 5, 50, 1]     # beyond every row, empty, the first timestamp only
    idx = grab.CagraIndex(dim, 32, vmm_max_bytes=1 << 30)
    idx.add(data[:n0], ts[:n0])
    idx.build()
    for n in (n0, n0 + n1):
        if n > n0:
            idx.insert(data[n0:n], ts[n0:n])
        ids, dist = idx.scan_range_batch(q, k, ws, we)
        eids, edist = oracle.bruteforce_topk(data[:n], q, k, filter_kind=oracle.FILTER_RANGE, ts=ts[:n], win_start=ws, win_end=we)
        assert np.array_equal(ids, eids)
        valid = ids >= 0
        assert np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid]) and (dist[~valid] == -1.0).all()
        assert (ids[:2] == -1).all() and (ids[2] >= 0).sum() == 7
    idx.close()
    # timestamps in no order
    ts2 = rng.permutation(ts[:n0])
    idx = grab.CagraIndex(dim, 32, vmm_max_bytes=1 << 30)
    idx.add(data[:n0], ts2)
    idx.build()
    ids, dist = idx.scan_range_batch(q, k, ws, we)
    eids, edist = oracle.bruteforce_topk(data[:n0], q, k, filter_kind=oracle.FILTER_RANGE, ts=ts2, win_start=ws, win_end=we)
    assert np.array_equal(ids, eids)
    idx.close()


def test_range_batches_scan_their_narrow_windows(oracle, grab):
    # set_scan_below: one call, the narrow windows scanned exactly, the wide ones searched on the graph as ever
    n, dim, k, nq = 8000, 64, 10, 400
    data = datasets.mixture(n, dim, 20, 3, 4)
    ts = np.arange(n, dtype=np.uint64) * 2
    q = datasets.mixture(nq, dim, 20, 3, 5)
    rng = np.random.default_rng(9)
    width = np.where(rng.random(nq) < 0.5, rng.integers(20, 300, nq), rng.integers(2000, 6000, nq)).astype(np.uint64)
    ws = rng.integers(0, 2 * n - 2 * int(width.max()), nq).astype(np.uint64)
    we = ws + 2 * width
    idx = grab.CagraIndex(dim, 32, vmm_max_bytes=1 << 30)
    idx.set_seed(5)
    idx.setQueryParams(64, 4, 0, 50, 12)
    idx.add(data, ts)
    idx.build()
    plain_ids, plain_dist = idx.query_range_batch(q, k, ws, we)
    idx.set_seed(5)
    idx.set_scan_below(0.05)                      # 400 rows
    ids, dist = idx.query_range_batch(q, k, ws, we)
    narrow = width <= 400
    assert narrow.any() and (~narrow).any()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=ts, win_start=ws, win_end=we)
    assert np.array_equal(ids[narrow], eids[narrow])
    assert np.array_equal(dist[narrow].view(np.uint32), edist[narrow].view(np.uint32))
    # the wide ones: a graph search of that half alone with the same generator state
    idx.set_scan_below(0.0)
    idx.set_seed(5)
    wide_ids, wide_dist = idx.query_range_batch(q[~narrow], k, ws[~narrow], we[~narrow])
    assert np.array_equal(ids[~narrow], wide_ids) and np.array_equal(dist[~narrow].view(np.uint32), wide_dist.view(np.uint32))
    assert datasets.recall(ids, eids) >= datasets.recall(plain_ids, eids)
    # all narrow / none narrow
    idx.set_scan_below(1.0)
    a, _ = idx.query_range_batch(q, k, ws, we)
    assert np.array_equal(a, eids)
    idx.close()


def test_window_scan_in_several_passes(oracle, grab):
    # the dense block is made in passes of at most 128 row tiles (16,384 queries) and at most 4 GiB: more queries than a
    # pass takes, and intervals so long that 16 row tiles already pass the 4 GiB
    n, dim, k = 60000, 32, 10
    data = datasets.unit_rows(n, dim, 61)
    d_data = grab.DeviceArray.from_numpy(data)
    ts = grab.DeviceArray.from_numpy(np.arange(n, dtype=np.uint64))
    nq = 20000
    q = datasets.unit_rows(nq, dim, 62)
    d_q = grab.DeviceArray.from_numpy(q)
    lo, hi = _intervals(n, nq, 50, 700, 63)
    ids, dist, _ = grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi)
    gids, gdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, filter_kind=grab.FILTER_RANGE, d_ts=ts,
                                          d_win_start=grab.DeviceArray.from_numpy(lo), d_win_end=grab.DeviceArray.from_numpy(hi))
    assert np.array_equal(ids, gids) and np.array_equal(dist.view(np.uint32), gdist.view(np.uint32))
    pick = np.arange(0, nq, 997)
    eids, _ = oracle.bruteforce_topk(data, q[pick], k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64),
                                     win_start=lo[pick], win_end=hi[pick])
    assert np.array_equal(ids[pick], eids)
    del d_data, d_q, ts

    n, nq = 1_000_000, 2100                      # 17 row tiles x 128 rows x ~600,000 columns x 4 bytes: 5 GB
    data = datasets.unit_rows(n, dim, 64)
    q = datasets.unit_rows(nq, dim, 65)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    ts = grab.DeviceArray.from_numpy(np.arange(n, dtype=np.uint64))
    lo, hi = _intervals(n, nq, 500000, 520000, 66)
    ids, dist, _ = grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi)
    gids, gdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, filter_kind=grab.FILTER_RANGE, d_ts=ts,
                                          d_win_start=grab.DeviceArray.from_numpy(lo), d_win_end=grab.DeviceArray.from_numpy(hi))
    assert np.array_equal(ids, gids) and np.array_equal(dist.view(np.uint32), gdist.view(np.uint32))


@pytest.mark.parametrize("n,dim,nq,k,metric,widths,kind", [
    (30000, 96, 1200, 10, 0, (5900, 9000), "mix"),     # ties between integer rows; narrow for short lists
    (30000, 96, 1200, 10, 0, (11000, 14000), "mix"),   # ... and wide enough
    (12001, 32, 1030, 128, 0, (1, 12001), "gauss"),    # the longest lists, intervals from one row to all
    (20000, 288, 1100, 16, 1, (6100, 15000), "unit"),  # an odd number of chunks of 32 dimensions
    (40000, 128, 1500, 40, 1, (200, 300), "unit"),     # narrow intervals, lists too long for stored values
    (8200, 64, 1100, 100, 0, (60, 140), "mix"),        # intervals shorter than k among them
    (9000, 64, 1100, 20, 0, (300, 4000), "far"),       # queries far longer than the rows: the way before this one
    (9000, 64, 1100, 20, 0, (300, 4000), "dup"),       # every row forty times: more ties than a list holds
])
def test_window_scan_on_f16_rows(oracle, grab, n, dim, nq, k, metric, widths, kind):
    make = {"mix": lambda m, s: datasets.mixture(m, dim, 12, 3, s), "unit": lambda m, s: datasets.unit_rows(m, dim, s)}.get(
        kind, lambda m, s: datasets.gaussian(m, dim, s))
    data, q = make(n, 4), make(nq, 7)
    if kind == "far":
        q *= np.float32(100.0)
    elif kind == "dup":
        data = np.ascontiguousarray(np.repeat(data[:n // 40], 40, axis=0)[:n])
    lo, hi = _intervals(n, nq, widths[0], widths[1], 3 * n + dim)
    lo[5], hi[5] = 17, 17
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, len(data), dim, metric)
    ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
    assert (grab.last_knn_f16_flop() > 0) == (kind != "far" and widths != (5900, 9000)) and grab.last_knn_bf16_flop() > 0
    base.close()
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=metric, filter_kind=oracle.FILTER_RANGE, ts=np.arange(len(data), dtype=np.uint64),
                                         win_start=lo, win_end=np.minimum(hi, np.uint64(len(data))))
    bad = np.flatnonzero((ids != eids).any(axis=1))
    assert bad.size == 0, f"queries {bad[:5]}: {ids[bad[0]]} vs {eids[bad[0]]} in [{lo[bad[0]]}, {hi[bad[0]]})"
    valid = ids >= 0
    assert np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])


@pytest.mark.parametrize("widths,on_f16", [((90000, 126000), True), ((127500, 140000), False)])
def test_window_scan_of_wide_intervals(oracle, grab, widths, on_f16):
    # one block of 64 at least is sampled: a list of 2048 then holds what five sampled values stand for, but for one query in
    # 10^4; intervals on the other side of the limit keep the way of rows as two bf16 halves
    n, dim, nq, k = 140000, 32, 1030, 10
    data, q = datasets.gaussian(n, dim, 4), datasets.gaussian(nq, dim, 7)
    lo, hi = _intervals(n, nq, widths[0], widths[1], 5)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, n, dim, 0)
    ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
    assert (grab.last_knn_f16_flop() > 0) == on_f16 and grab.last_knn_bf16_flop() > 0
    if on_f16:
        assert grab.last_knn_stats()[1] <= 5
    base.close()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo,
                                         win_end=np.minimum(hi, np.uint64(n)))
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


@pytest.mark.parametrize("edge,dim,k", [(1 << 26, 32, 10), (1 << 26, 32, 40), (1 << 28, 32, 40), (1 << 29, 4, 10)])
def test_scans_beyond_67_million_rows(oracle, grab, edge, dim, k):
    # 2^26 columns are what the queue's words once held of a row's number, 2^28 the rows that one launch packs, 2^29 those whose
    # norms one launch took (rows of 4: fp32 instructions): intervals and buckets on either side of that row and across it, short
    # ones (every column listed) and long ones
    nq = 300
    first, n = edge - 20000, edge + 30000
    data, q = datasets.gaussian(n - first, dim, 4), datasets.gaussian(nq, dim, 7)
    d_data, d_q = grab.DeviceArray((n, dim), np.float32), grab.DeviceArray.from_numpy(q)
    d_data.fill_bytes(0)
    grab.check(grab.lib.grab_copy_to_device(C.c_void_p(d_data.ptr + first * dim * 4), data.ctypes.data_as(C.c_void_p), C.c_size_t(data.nbytes)))
    rng = np.random.default_rng(k)
    width = np.where(np.arange(nq) % 3 == 0, rng.integers(1, 257, nq), rng.integers(18000, 20000, nq))
    lo = np.where(np.arange(nq) % 2 == 0, rng.integers(edge, n - width), np.maximum(edge - rng.integers(0, width + 1), first)).astype(np.uint64)
    hi = np.minimum(lo + width.astype(np.uint64), np.uint64(n))
    base = grab.ScanBase(d_data, n, dim, 0)
    ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
    assert grab.last_knn_stats()[1] <= 3 and (grab.last_knn_f16_flop() > 0) == (dim % 32 == 0)  # the candidates prove the answers
    own = np.arange(n - first, dtype=np.uint64)
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=own, win_start=lo - np.uint64(first), win_end=hi - np.uint64(first))
    valid = eids >= 0
    assert np.array_equal(ids, np.where(valid, eids + first, -1)) and np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])
    offsets = np.array([first, edge - 9000, edge - 100, edge + 120, edge + 200, edge + 15000, n], np.uint64)
    labels = (np.searchsorted(offsets, own + np.uint64(first), side="right") - 1).astype(np.uint8)
    masks = rng.integers(1, 64, nq).astype(np.uint64)
    masks[:30] = np.uint64(1 << 3)  # a bucket of 80 rows
    ids, dist, _ = base.bucket_topk(offsets, d_q, nq, k, masks)
    base.close()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks)
    valid = eids >= 0
    assert np.array_equal(ids, np.where(valid, eids + first, -1)) and np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])


@pytest.mark.parametrize("run,k,widths", [(10, 10, (8000, 12000)), (40, 10, (40000, 60000)), (200, 40, (40000, 60000)), (1, 10, None)])
def test_window_scan_of_rows_that_resemble_their_neighbours(oracle, grab, run, k, widths):
    # rows in runs (frames of a scene), the query's run inside its interval; last, intervals of 1500 among long ones: what a query is
    # bounded by is sampled from all of its interval, so that next to no query's candidates fail to prove the answer
    n, dim, nq = 140000, 32, 1030
    rng = np.random.default_rng(run)
    scenes = datasets.gaussian((n + run - 1) // run, dim, 4) * np.float32(8.0)
    data = np.repeat(scenes, run, axis=0)[:n] + datasets.gaussian(n, dim, 5)
    own = rng.integers(0, n, nq)
    q = data[own] + datasets.gaussian(nq, dim, 6)
    width = rng.integers(widths[0], widths[1], nq) if widths else np.where(np.arange(nq) % 2, 1500, 90000)
    lo = np.clip(own - (rng.random(nq) * width).astype(np.int64), 0, n - width).astype(np.uint64)
    hi = lo + width.astype(np.uint64)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, n, dim, 0)
    ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
    assert grab.last_knn_stats()[1] <= 5 and grab.last_knn_f16_flop() > 0
    base.close()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


@pytest.mark.parametrize("nq,width,k,on_f16", [(1, 11000, 10, False), (1, 11400, 16, True), (2, 10500, 10, False), (2, 11300, 10, True), (300, 9000, 16, False),
                                               (300, 11000, 10, True), (3000, 2999, 16, False), (3, 300, 17, True)])
def test_window_scan_of_few_queries(oracle, grab, nq, width, k, on_f16):
    # narrow intervals with short lists keep the way of stored values, the longer the fewer the queries and the shorter the rows
    n, dim = 30000, 64
    data, q = datasets.gaussian(n, dim, 4), datasets.gaussian(nq, dim, 7)
    lo, hi = _intervals(n, nq, width, width, nq)
    base = grab.ScanBase(grab.DeviceArray.from_numpy(data), n, dim, 0)
    ids, dist, _ = base.window_topk(grab.DeviceArray.from_numpy(q), nq, k, lo, hi)
    assert (grab.last_knn_f16_flop() > 0) == on_f16 and grab.last_knn_bf16_flop() > 0
    base.close()
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


@pytest.mark.parametrize("nq,k,width", [(1_300_000, 17, 300), (70_000, 17, 60_000)])
def test_window_scan_of_many_queries_takes_bounded_memory(oracle, grab, nq, k, width):
    # lists of 8 KB a query, then some thousand sampled values a query: in passes of 4 GiB, whose scratch the base keeps
    n, dim = 250_000, 32
    data, q = datasets.gaussian(n, dim, 4), datasets.gaussian(nq, dim, 7)
    lo, hi = _intervals(n, nq, width - 50, width, nq)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    out = (grab.DeviceArray((nq, k), np.int64), grab.DeviceArray((nq, k), np.float32))
    base = grab.ScanBase(d_data, n, dim, 0)
    free = grab.device_memory()[0]
    base.window_topk(d_q, nq, k, lo, hi, d_out=out)
    assert grab.last_knn_f16_flop() > 0 and grab.last_knn_stats()[1] <= 20
    time.sleep(1.0)  # the first call's scratch is given back, which the driver takes its time over
    assert free - grab.device_memory()[0] < 5 << 30
    base.close()
    pick = np.concatenate([[0, nq // 2 - 1, nq // 2, nq - 1], np.random.default_rng(1).integers(0, nq, 400)])
    ids, dist = out[0].numpy()[pick], out[1].numpy()[pick]
    eids, edist = oracle.bruteforce_topk(data, q[pick], k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo[pick], win_end=hi[pick])
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


def test_window_scan_of_many_queries_half_of_them_without_a_row(oracle, grab):
    # lists of 560,000 queries are more than a pass takes; of the two that it is cut into one has no row at all
    n, dim, nq, k = 20000, 32, 1_120_000, 17
    data, q = datasets.gaussian(n, dim, 4), datasets.gaussian(nq, dim, 7)
    lo, hi = _intervals(n, nq, 250, 300, 5)
    hi[:nq // 2] = lo[:nq // 2]
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    out = (grab.DeviceArray((nq, k), np.int64), grab.DeviceArray((nq, k), np.float32))
    base = grab.ScanBase(d_data, n, dim, 0)
    base.window_topk(d_q, nq, k, lo, hi, d_out=out)
    assert grab.last_knn_f16_flop() > 0
    base.close()
    ids, dist = out[0].numpy(), out[1].numpy()
    assert (ids[:nq // 2] == -1).all() and (dist[:nq // 2] == np.float32(3.40282e38)).all()
    pick = np.concatenate([[nq // 2, nq - 1], np.random.default_rng(1).integers(nq // 2, nq, 400)])
    eids, edist = oracle.bruteforce_topk(data, q[pick], k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo[pick], win_end=hi[pick])
    assert np.array_equal(ids[pick], eids) and np.array_equal(dist[pick].view(np.uint32), edist.view(np.uint32))


def test_scan_base_where_the_rows_as_bf16_halves_find_no_room(oracle, grab):
    # narrow intervals would have the halves made: where the memory is not there they are scanned on f16 rows, those that f16 rows
    # do not take on the rows as they are, nothing is left allocated, and with the memory back the halves are made
    n, dim, nq, k = 2_000_000, 128, 60, 10
    data, q = np.random.default_rng(4).standard_normal((n, dim), np.float32), datasets.gaussian(nq, dim, 7)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, n, dim, 0)
    taken = []
    for size in (4 << 30, 256 << 20):
        try:
            while True:
                taken.append(grab.DeviceArray((size,), np.uint8))
        except grab.GrabError:
            pass
    for _ in range(2):  # 512 to 768 MB: the halves take 1024
        taken.pop().free()

    def scan(widths, f16, halves, seed=3):
        lo, hi = _intervals(n, nq, widths[0], widths[1], seed)
        lo, hi = lo % np.uint64(1000), hi - lo + lo % np.uint64(1000)
        ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
        assert (grab.last_knn_f16_flop() > 0) == f16 and (grab.last_knn_bf16_flop() > 0) == (f16 or halves)
        own = slice(0, int(hi.max()))
        eids, edist = oracle.bruteforce_topk(data[own], q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(own.stop, dtype=np.uint64), win_start=lo, win_end=hi)
        assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
        return grab.device_memory()[0]

    scan((2000, 3000), True, False)
    free = scan((127500, 150000), False, False)  # (the base's block is as large as it gets)
    for _ in range(3):
        scan((2000, 3000), True, False)
        now = scan((127500, 150000), False, False)
    assert now > free - (16 << 20)  # norms of each of the six calls would be 48 MB
    for t in taken:
        t.free()
    scan((2000, 3000), False, True)
    scan((127500, 150000), False, True)
    base.close()


def test_scan_base_of_rows_that_are_not_finite_keeps_no_f16_rows(grab):
    n, dim = 4_000_000, 32
    d_data = grab.DeviceArray((n, dim), np.float32)
    d_data.fill_bytes(0)
    free = grab.device_memory()[0]
    base = grab.ScanBase(d_data, n, dim, 0)
    kept = free - grab.device_memory()[0]
    base.close()
    nan = np.full(dim, np.nan, np.float32)
    grab.check(grab.lib.grab_copy_to_device(C.c_void_p(d_data.ptr + 5 * dim * 4), nan.ctypes.data_as(C.c_void_p), C.c_size_t(nan.nbytes)))
    free = grab.device_memory()[0]
    base = grab.ScanBase(d_data, n, dim, 0)
    halves = free - grab.device_memory()[0]
    base.close()
    assert kept > 0 and halves < n * (dim * 4 + 4) + (64 << 20)  # halves and norms, and no more


@pytest.mark.parametrize("nq,k,widths", [(1, 10, (20000, 25000)), (300, 10, (9000, 25000)), (1100, 40, (100, 25000))])
def test_scans_of_rows_far_from_the_origin(oracle, grab, nq, k, widths):
    # a hundred standard deviations in every coordinate: the rows are centred, and so is what the proof allows for
    n, dim = 25000, 128
    data, q = datasets.gaussian(n, dim, 4) + np.float32(100.0), datasets.gaussian(nq, dim, 7) + np.float32(100.0)
    lo, hi = _intervals(n, nq, widths[0], widths[1], nq)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = grab.ScanBase(d_data, n, dim, 0)
    ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
    assert grab.last_knn_f16_flop() > 0 and grab.last_knn_stats()[1] <= 3
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
    offsets = np.array([0, 3000, 3100, 15000, n], np.uint64)
    masks = np.random.default_rng(nq).integers(1, 16, nq).astype(np.uint64)
    ids, dist, _ = base.bucket_topk(offsets, d_q, nq, k, masks)
    assert grab.last_knn_f16_flop() > 0 and grab.last_knn_stats()[1] <= 3
    base.close()
    labels = np.repeat(np.arange(4, dtype=np.uint8), np.diff(offsets.astype(np.int64)))
    eids, edist = oracle.bruteforce_topk(data, q, k, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks)
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))


@pytest.mark.parametrize("nq,one_shot", [(60, False), (2000, False), (2000, True)])
def test_scans_whose_f16_rows_do_not_prove_all_queries(oracle, grab, nq, one_shot):
    # inner products of unit rows in tight clusters: what rounding to f16 moved them by hides the order of some. Those queries go over the
    # rows as they are, which proves them, or over bf16 halves where they are many, which leaves some to be scored against every row
    n, dim, k = 30000, 128, 32
    rng = np.random.default_rng(5)
    data = datasets.gaussian(60, dim, 4)[rng.integers(0, 60, n)] * np.float32(10.0) + datasets.gaussian(n, dim, 6) * np.float32(0.25)
    data /= np.linalg.norm(data, axis=1, keepdims=True)
    q = data[rng.integers(0, n, nq)].copy()
    lo, hi = _intervals(n, nq, 6000, 7000, nq)
    hi[::50] = lo[::50]
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    base = None if one_shot else grab.ScanBase(d_data, n, dim, 1)
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=1, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
    for _ in range(2):
        ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi) if base else grab.window_scan_topk(d_data, n, dim, d_q, nq, k, lo, hi, metric=1)
        assert grab.last_knn_f16_flop() > 0 and grab.last_knn_stats()[1] > 0 and grab.last_knn_exact_rows() <= (grab.last_knn_stats()[1] if nq >= 128 else 0)
        valid = eids >= 0
        assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])
    offsets = np.array([0, 6000, 6100, 15000, n], np.uint64)
    masks = np.random.default_rng(nq).integers(0, 16, nq).astype(np.uint64)
    ids, dist, _ = (base.bucket_topk(offsets, d_q, nq, k, masks) if base else
                    grab.bucket_scan_topk(d_data, n, dim, offsets, d_q, nq, k, masks, metric=1))
    assert grab.last_knn_f16_flop() > 0 and grab.last_knn_stats()[1] > 0
    labels = np.repeat(np.arange(4, dtype=np.uint8), np.diff(offsets.astype(np.int64)))
    eids, edist = oracle.bruteforce_topk(data, q, k, metric=1, filter_kind=oracle.FILTER_MASK, labels=labels, masks=masks)
    valid = eids >= 0
    assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32)[valid], edist.view(np.uint32)[valid])


def test_scan_base_of_rows_that_point_one_way(oracle, grab):
    # a hundred deviations off zero in every coordinate: inner products on bf16 halves from the start, squared distances on f16 rows
    n, dim, nq, k = 30000, 128, 300, 10
    data, q = datasets.gaussian(n, dim, 4) + np.float32(100.0), datasets.gaussian(nq, dim, 7) + np.float32(100.0)
    lo, hi = _intervals(n, nq, 13000, 14000, nq)
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    for metric in (0, 1):
        base = grab.ScanBase(d_data, n, dim, metric)
        ids, dist, _ = base.window_topk(d_q, nq, k, lo, hi)
        assert (grab.last_knn_f16_flop() > 0) == (metric == 0) and grab.last_knn_bf16_flop() > 0
        base.close()
        eids, edist = oracle.bruteforce_topk(data, q, k, metric=metric, filter_kind=oracle.FILTER_RANGE, ts=np.arange(n, dtype=np.uint64), win_start=lo, win_end=hi)
        assert np.array_equal(ids, eids) and np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
