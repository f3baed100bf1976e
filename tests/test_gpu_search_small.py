"""Small batches: the kernel made for the time of one query, where its shapes change - 1024 / 512 threads, one to sixteen
queue blocks, candidates merged beside the expansion or before it, rows that are no whole rounds of loads - and the general
kernel for what that one refuses, against the oracle."""
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
    (4, 64, 32, 20, 128, 32, 13, True), (2, 64, 4, 0, 128, 32, 13, False), (2, 64, 4, 1, 128, 32, 13, False), (6, 10, 2, 45, 128, 32, 12, False),
    (300, 64, 32, 20, 128, 32, 13, True), (3, 1000, 40, 20, 96, 32, 14, False),  # more neighbours than threads
    (2, 64, 18, 30, 128, 32, 13, False), (2, 64, 19, 30, 128, 32, 13, True),     # the last width it takes, and the first it does not
    # what that kernel refuses: 1024 threads of the general one, merges split over the waves or plain, tables in LDS or not
    (3, 1100, 4, 40, 128, 32, 13, False), (256, 1030, 4, 33, 96, 32, 13, True), (257, 1100, 4, 20, 96, 32, 13, True),
    (5, 64, 64, 12, 128, 32, 16, True), (2, 900, 100, 10, 128, 32, 15, False)])
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


@pytest.mark.parametrize("bitlen", [4, 6, 8, 10])
@pytest.mark.parametrize("nq", [3, 300, 513])
@pytest.mark.parametrize("how", ["all", "filter_first", "filter_after"])
def test_visited_set_takes_its_size_and_no_more(grab, oracle, how, nq, bitlen):
    # which ids a set that fills up refuses depends on their order, how many it takes does not, whatever kernel runs:
    # up to the first rebuild (30 iterations) 2^bitlen ids are scored, and the others counted as refused
    data, graph, d_data, d_graph = case(oracle, grab, 128, 32)
    n, cap = data.shape[0], 1 << bitlen
    d_q = grab.DeviceArray.from_numpy(datasets.mixture(nq, 128, 20, 10, 14))
    seeds = np.stack([np.random.default_rng(i).permutation(n)[:128] for i in range(nq)]).astype(np.uint32)
    dev = dict(d_seeds=grab.DeviceArray.from_numpy(seeds), n_provided=128)
    if how != "all":  # a window that admits every row
        dev.update(filter_kind=grab.FILTER_ID_RANGE, win=(0, n), flags=grab.FLAG_FILTER_FIRST if how == "filter_first" else 0)
    for iters in (0, 30):
        _, _, ctr, _ = grab.search_ex(d_data, d_graph, n, 128, 32, d_q, nq, 10, 128, 4, iters, bitlen, 128, 7, want_counters=True, **dev)
        scored, refused = ctr[:, 1] + ctr[:, 4], ctr[:, 5]
        assert (ctr[:, 1] == min(cap, 128)).all()
        assert (scored[refused > 0] == cap).all() and (scored <= cap).all(), (iters, scored.min(), scored.max())
        if iters == 0:
            assert (refused == max(128 - cap, 0)).all()
        else:
            assert (refused > 0).any() or bitlen == 10


@pytest.mark.parametrize("nq", [2, 513])
@pytest.mark.parametrize("dim", [36, 96, 104])
def test_products_that_vanish_keep_their_sign(oracle, grab, dim, nq):
    # every product underflows: a row's inner product is -0 or +0, which differ in the result and in the order
    n, k = 300, 10
    rng = np.random.default_rng(dim)
    data = (np.float32(1e-30) * rng.choice(np.float32([-1, 1]), (n, 1))) * np.ones((1, dim), np.float32)
    q = np.full((nq, dim), 1e-30, np.float32)
    graph = rng.integers(0, n, (n, 32)).astype(np.uint32)
    seeds = np.tile(np.arange(64, dtype=np.uint32), (nq, 1))
    d_data, d_q = grab.DeviceArray.from_numpy(data), grab.DeviceArray.from_numpy(q)
    eids, edist, _ = oracle.search(data, graph, q, k, 64, 2, 20, 13, 64, 5, metric=1, seeds=seeds)
    ids, dist, _, _ = grab.search_ex(d_data, grab.DeviceArray.from_numpy(graph), n, dim, 32, d_q, nq, k, 64, 2, 20, 13, 64, 5, metric=1,
                                     d_seeds=grab.DeviceArray.from_numpy(seeds), n_provided=64)
    assert np.array_equal(dist.view(np.uint32), edist.view(np.uint32)) and np.array_equal(ids, eids)
    # the exact scan re-scores its candidates in the same order of sums
    bids, bdist, _ = grab.bruteforce_topk(d_data, n, dim, d_q, nq, k, metric=1)
    xids, xdist = oracle.bruteforce_topk(data, q, k, metric=1)
    assert np.array_equal(bdist.view(np.uint32), xdist.view(np.uint32)) and np.array_equal(bids, xids)
