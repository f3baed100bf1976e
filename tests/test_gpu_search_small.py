"""Small batches: the kernel made for the time of one query, where its shapes change - 1024 / 512 threads, one to sixteen
queue blocks, candidates merged beside the expansion or before it, rows that are no whole rounds of loads - against the oracle."""
import numpy as np
import pytest

import datasets

pytestmark = pytest.mark.gpu

CASES = {}


def case(oracle, grab, dim, deg):
    if (dim, deg) not in CASES:
        data = datasets.mixture(3000, dim, 20, 10, 11)
        graph = oracle.optimize(oracle.knn_graph(data, 2 * deg), deg)
        CASES[dim, deg] = data, graph, grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(graph)
    return CASES[dim, deg]


@pytest.mark.parametrize("nq,itopk,width,iters,dim,deg,bitlen,filtered", [
    (1, 64, 4, 50, 128, 32, 13, False), (3, 256, 6, 50, 128, 32, 13, False), (256, 65, 4, 40, 96, 32, 12, True),
    (257, 128, 4, 40, 96, 32, 12, True), (512, 64, 1, 35, 100, 32, 11, False), (513, 64, 4, 35, 100, 32, 12, False),
    (5, 300, 4, 62, 132, 24, 13, False), (7, 1000, 3, 31, 32, 24, 14, True), (9, 64, 20, 40, 32, 24, 17, False),
    (4, 64, 32, 20, 128, 32, 13, True), (2, 64, 4, 0, 128, 32, 13, False), (2, 64, 4, 1, 128, 32, 13, False), (6, 10, 2, 45, 128, 32, 12, False)])
def test_small_batch_matches_oracle(oracle, grab, nq, itopk, width, iters, dim, deg, bitlen, filtered):
    data, graph, d_data, d_graph = case(oracle, grab, dim, deg)
    n, k = data.shape[0], 10
    q = datasets.mixture(nq, dim, 20, 10, 12)
    kw, dev = {}, {}
    if filtered:
        ws, we = datasets.windows(n, nq, 0.3, 13)
        kw = dict(filter_kind=oracle.FILTER_ID_RANGE, win_start=ws, win_end=we, flags=oracle.FLAG_FILTER_FIRST)
        dev = dict(filter_kind=grab.FILTER_ID_RANGE, d_win_start=grab.DeviceArray.from_numpy(ws), d_win_end=grab.DeviceArray.from_numpy(we),
                   flags=grab.FLAG_FILTER_FIRST)
    seeds = min(itopk, 64)
    eids, edist, ectr = oracle.search(data, graph, q, k, itopk, width, iters, bitlen, seeds, 0x9E3779B9, **kw)
    assert ectr[:, 5].sum() == 0  # a table that fills up is order-dependent
    ids, dist, ctr, _ = grab.search_ex(d_data, d_graph, n, dim, deg, grab.DeviceArray.from_numpy(q), nq, k, itopk, width, iters, bitlen, seeds,
                                       0x9E3779B9, want_counters=True, **dev)
    assert np.array_equal(ids, eids)
    assert np.array_equal(dist.view(np.uint32), edist.view(np.uint32))
    assert np.array_equal(ctr, ectr)
