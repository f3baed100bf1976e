"""The work that users of the index have it do, as cases that can be timed.

A case names one path through the public entry points and its sizes.  Base rows are the mixture of the benchmark
(1000 centroids in [0,128]^dim, sigma 16, rounded to integers in [0,255]) for squared L2 and unit rows for the inner
product; queries are fresh rows of the same distribution, windows lie anywhere in the timestamps, labels follow a Zipf law.

  query        index handle, host arrays in and out, the calls of the reference's classes: CagraIndex.query,
               query_range (one window for the batch) or query_local (one bucket of the time-partitioned graph)
  batch        index handle, host arrays, a window per query: query_range_batch with the entry-point layer
  search       device arrays: unfiltered search
  range        device arrays: seeds listed from the entry-point layer, then the search inside every query's window;
               timestamps in row order, or in any order (the interval is tested on a row's place in timestamp order)
  window_scan  exact top-k inside narrow windows over a prepared base, device arrays
  bucket_scan  exact top-k inside sets of buckets over a prepared base, device arrays
  index        an index from host arrays: create, add, build
  build        device arrays: kNN graph, then the pruned graph
  insert       device arrays: rows inserted 64 at a time, each step into the graph that the steps before it left
"""
import importlib
import math

import numpy as np
import torch

grab = importlib.import_module("grab-anns_amd")

DEV = "cuda"


def listed():
    return [
        # one user waiting for one answer: latency of a call with the handle's default parameters
        dict(name="query_1", op="query", filter="none", n=100_000, dim=128, nq=1, k=10, itopk=256, width=6, bitlen=13, degree=64),
        # a small batch that shares a window, the reference's query_range
        dict(name="query_window_100", op="query", filter="window", n=200_000, dim=96, nq=100, k=10, itopk=128, width=4, bitlen=13, degree=64),
        # a batch inside one bucket of the time-partitioned graph, the reference's query_local
        dict(name="query_bucket_777", op="query", filter="bucket", n=60_000, dim=256, nq=777, k=20, itopk=128, width=4, bitlen=13, degree=64),
        # an application that keeps its vectors in host memory and sends batches of range queries
        dict(name="batch_10k", op="batch", n=300_000, dim=128, nq=10_000, k=10, itopk=64, selectivity=0.1, degree=64),
        # the unfiltered search of the configuration with a million rows
        dict(name="search_10k", op="search", n=1_000_000, dim=128, nq=10_000, k=10, itopk=64, width=4, bitlen=13, degree=64),
        # the benchmark's headline: 10 % windows, everything in device memory
        dict(name="range_10k", op="range", n=1_000_000, dim=128, nq=10_000, k=10, itopk=64, selectivity=0.1, ordered=True, degree=64),
        # narrow windows, where an exact scan is the better tool
        dict(name="window_scan_10k", op="window_scan", n=1_000_000, dim=128, nq=10_000, k=10, selectivity=0.01, metric="l2"),
        # label sets over long embedding rows, inner product, a ragged batch
        dict(name="bucket_scan_4999", op="bucket_scan", n=200_000, dim=768, nq=4999, k=10, labels=64, metric="ip"),
        # the smallest configuration, from host arrays to an index
        dict(name="index_10k", op="index", n=10_000, dim=128, degree=64, metric="l2"),
        # the graph of the configuration with a million rows
        dict(name="build_1m", op="build", n=1_000_000, dim=128, degree=64, metric="l2"),
        # long embedding rows, inner product, a ragged row count
        dict(name="build_ip_768", op="build", n=100_003, dim=768, degree=64, metric="ip"),
        # a stream of new rows, 64 at a time with a short last step
        dict(name="insert_1000", op="insert", n=200_000, dim=128, rows=1000, degree=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["query", "query", "batch", "search", "range", "range", "window_scan", "bucket_scan", "index", "build", "build", "insert"])
    dim = rng.choice([96, 100, 128, 128, 256, 384, 768])
    most = int(1.28e8 / dim)  # rows whose vectors take 512 MB
    degree = rng.choice([32, 64, 64])
    if op == "query":
        return dict(op=op, filter=rng.choice(["none", "window", "bucket"]), n=_log_int(rng, 20_000, min(most, 200_000)), dim=dim,
                    nq=_log_int(rng, 1, 2000), k=rng.choice([1, 10, 20, 50]), itopk=rng.choice([64, 128, 256]), width=rng.choice([4, 6]),
                    bitlen=13, degree=degree)
    if op == "batch":
        return dict(op=op, n=_log_int(rng, 50_000, min(most, 300_000)), dim=dim, nq=_log_int(rng, 300, 10_000), k=10,
                    itopk=rng.choice([64, 128]), selectivity=rng.choice([0.05, 0.1, 0.3]), degree=degree)
    if op == "search":
        return dict(op=op, n=_log_int(rng, 50_000, min(most, 1_000_000)), dim=dim, nq=_log_int(rng, 300, 10_000), k=rng.choice([10, 50]),
                    itopk=rng.choice([64, 128, 256]), width=4, bitlen=13, degree=degree)
    if op == "range":
        return dict(op=op, n=_log_int(rng, 50_000, min(most, 1_000_000)), dim=dim, nq=_log_int(rng, 300, 10_000), k=10,
                    itopk=rng.choice([64, 64, 128]), selectivity=rng.choice([0.05, 0.1, 0.2, 0.5]), ordered=rng.random() < 0.7, degree=degree)
    if op == "window_scan":
        return dict(op=op, n=_log_int(rng, 50_000, min(most, 1_000_000)), dim=dim, nq=_log_int(rng, 100, 10_000), k=rng.choice([10, 16, 40]),
                    selectivity=round(math.exp(rng.uniform(math.log(0.001), math.log(0.04))), 4), metric="l2" if dim <= 256 else rng.choice(["l2", "ip"]))
    if op == "bucket_scan":
        return dict(op=op, n=_log_int(rng, 20_000, min(most, 200_000)), dim=dim, nq=_log_int(rng, 100, 5000), k=10,
                    labels=rng.choice([16, 33, 64]), metric="ip" if dim > 256 else rng.choice(["l2", "ip"]))
    if op == "index":
        return dict(op=op, n=_log_int(rng, 2000, 50_000), dim=dim, degree=degree, metric="ip" if dim > 256 else "l2")
    if op == "build":
        cap = 100_000 if dim % 32 and dim > 128 else int(1_000_000 * math.sqrt(128 / max(dim, 128)) * 0.4)
        return dict(op=op, n=_log_int(rng, 10_000, cap), dim=dim, degree=degree, metric="ip" if dim > 256 else "l2")
    return dict(op=op, n=_log_int(rng, 20_000, min(most, 200_000)), dim=dim, rows=_log_int(rng, 64, 1000), degree=degree)


# ---- inputs --------------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _mixture(g, n, dim, centroids):
    which = torch.randint(0, centroids.shape[0], (n,), generator=g, device=DEV)
    x = torch.randn(n, dim, generator=g, device=DEV)
    return x.mul_(16.0).add_(centroids[which]).clamp_(0.0, 255.0).round_()


def _unit(g, n, dim):
    x = torch.randn(n, dim, generator=g, device=DEV)
    return x.div_(x.norm(dim=1, keepdim=True))


def _rows(case, seed, *counts):
    """Row sets of the case's distribution (the base first), from the seed alone."""
    g = _gen(seed)
    if case.get("metric", "l2") == "ip":
        return [_unit(g, c, case["dim"]) for c in counts]
    cent = torch.rand(1000, case["dim"], generator=g, device=DEV) * 128.0
    return [_mixture(g, c, case["dim"], cent) for c in counts]


def _windows(seed, n, nq, fraction):
    """One window per query, as host arrays of row ids / timestamps."""
    w = max(1, round(n * fraction))
    lo = np.random.default_rng(seed).integers(0, n - w + 1, nq).astype(np.uint64)
    return lo, lo + np.uint64(w)


def _metric(case):
    return grab.METRIC_IP if case.get("metric") == "ip" else grab.METRIC_L2


def _dev(a):
    """A host array of unsigned words as a device tensor with the same bits."""
    signed = {np.dtype(np.uint64): np.int64, np.dtype(np.uint32): np.int32}[a.dtype]
    return torch.from_numpy(a.view(signed)).to(DEV)


class _Tensor:
    """What torch needs to see a device array of the package as a tensor, without a copy (unsigned words as signed ones)."""

    def __init__(self, arr):
        self.arr = arr
        kind = {"f": "f", "u": "i", "i": "i"}[arr.dtype.kind]
        self.__cuda_array_interface__ = {"shape": arr.shape, "typestr": f"<{kind}{arr.dtype.itemsize}", "data": (arr.ptr, False), "version": 2}


def _tensor(arr):
    return torch.as_tensor(_Tensor(arr), device=DEV)


def _graph(x, n, dim, degree, metric):
    knn, _ = grab.generate_knn_graph(x.data_ptr(), n, dim, max(128, 2 * degree), metric)
    return grab.build_graph(x.data_ptr(), n, knn, max(128, 2 * degree), degree)


def _outputs(nq, k):
    out = (grab.DeviceArray((nq, k), np.int64), grab.DeviceArray((nq, k), np.float32))
    return out, (_tensor(out[0]), _tensor(out[1]))


def _visited_bits(n_seeds, degree, selectivity):
    """Slots for 1.25 times the in-window ids that 30 iterations of four parents can add, as in the benchmark."""
    need = 1.25 * (n_seeds + 30 * 4 * degree * selectivity)
    return min(13, max(8, math.ceil(math.log2(need))))


def _entry_groups(samples):
    return max(16, min(768, samples // 85))


def prepare(case, seed):
    s = dict(case)
    n, dim, op = case["n"], case["dim"], case["op"]
    torch.cuda.synchronize()
    if op == "query":
        base, q = _rows(case, seed, n, case["nq"])
        partitioned = case["filter"] == "bucket"
        idx = grab.CagraIndex(dim, case["degree"], vmm_max_bytes=4 << 30, local_degree=case["degree"] * 3 // 4 if partitioned else 0)
        idx.set_seed(seed)
        idx.setQueryParams(case["itopk"], case["width"], 0, 50, case["bitlen"])
        buckets = 20
        ts = np.arange(n, dtype=np.uint64) * np.uint64(buckets) // np.uint64(n) if partitioned else np.arange(n, dtype=np.uint64)
        idx.add(base.cpu().numpy(), ts)
        idx.build_partitioned() if partitioned else idx.build()
        s["idx"], s["q"] = idx, q.cpu().numpy()
        s["window"] = [int(w[0]) for w in _windows(seed + 1, n, 1, 0.1)]
        s["bucket"] = seed % buckets
    elif op == "batch":
        base, q = _rows(case, seed, n, case["nq"])
        samples = max(1024, n // 16)
        idx = grab.CagraIndex(dim, case["degree"], vmm_max_bytes=4 << 30)
        idx.set_seed(seed)
        idx.set_flags(grab.FLAG_FILTER_FIRST)
        idx.setQueryParams(case["itopk"], 4, 0, 50, _visited_bits(32, case["degree"], case["selectivity"]))
        idx.set_entry_layer(samples, 16)
        idx.set_entry_groups(_entry_groups(samples), 16, 16)
        idx.set_entry_list(32)
        idx.add(base.cpu().numpy(), np.arange(n, dtype=np.uint64))
        idx.build()
        s["idx"], s["q"], s["win"] = idx, q.cpu().numpy(), _windows(seed + 1, n, case["nq"], case["selectivity"])
        idx.query_range_batch(s["q"][:16], case["k"], s["win"][0][:16], s["win"][1][:16])  # a server primes its index before it takes queries
    elif op == "search":
        s["base"], s["q"] = _rows(case, seed, n, case["nq"])
        torch.cuda.synchronize()
        s["graph"] = _graph(s["base"], n, dim, case["degree"], _metric(case))
        s["out"], s["result"] = _outputs(case["nq"], case["k"])
        s["mask"] = seed * 2654435761 & 0xFFFFFFFF
    elif op == "range":
        s["base"], s["q"] = _rows(case, seed, n, case["nq"])
        nq, degree = case["nq"], case["degree"]
        lo, hi = _windows(seed + 1, n, nq, case["selectivity"])
        s["lo"], s["hi"] = _dev(lo), _dev(hi)
        s["ids"] = [torch.empty(nq, dtype=torch.int64, device=DEV) for _ in range(2)]
        s["seeds"] = torch.empty(nq, 32, dtype=torch.int32, device=DEV)
        samples = max(1024, n // 16)
        if case["ordered"]:
            s["ts"] = torch.arange(n, dtype=torch.int64, device=DEV)
            torch.cuda.synchronize()
            s["graph"] = _graph(s["base"], n, dim, degree, _metric(case))
            s["layer"] = grab.EntryLayer(s["base"].data_ptr(), n, dim, samples, d_ts=s["ts"].data_ptr())
        else:
            by_ts = torch.randperm(n, generator=_gen(seed + 2), device=DEV)
            rank = torch.empty(n, dtype=torch.int32, device=DEV)
            rank[by_ts] = torch.arange(n, dtype=torch.int32, device=DEV)
            s["rank"], s["by_ts"] = rank, by_ts.to(torch.int32)
            s["sorted_ts"] = torch.arange(n, dtype=torch.int64, device=DEV)
            s["ts"] = rank.to(torch.int64)
            torch.cuda.synchronize()
            s["graph"] = _graph(s["base"], n, dim, degree, _metric(case))
            s["graph_rank"] = grab.neighbor_ranks(s["graph"], rank.data_ptr(), n, degree)
            s["layer"] = grab.EntryLayer(s["base"].data_ptr(), n, dim, samples, d_ids_by_ts=s["by_ts"].data_ptr(), d_ts=s["ts"].data_ptr())
        s["layer"].build_groups(_entry_groups(samples), niter=10, seed=1)
        s["out"], s["result"] = _outputs(nq, case["k"])
        s["bitlen"] = _visited_bits(32, degree, case["selectivity"])
        s["mask"] = seed * 2654435761 & 0xFFFFFFFF
    elif op == "window_scan":
        s["base"], s["q"] = _rows(case, seed, n, case["nq"])
        torch.cuda.synchronize()
        s["scan"] = grab.ScanBase(s["base"].data_ptr(), n, dim, _metric(case))
        s["win"] = _windows(seed + 1, n, case["nq"], case["selectivity"])
        s["out"], s["result"] = _outputs(case["nq"], case["k"])
    elif op == "bucket_scan":
        s["base"], s["q"] = _rows(case, seed, n, case["nq"])
        torch.cuda.synchronize()
        s["scan"] = grab.ScanBase(s["base"].data_ptr(), n, dim, _metric(case))
        rng, labels, nq = np.random.default_rng(seed + 1), case["labels"], case["nq"]
        share = np.cumsum(1.0 / np.arange(1, labels + 1) ** 1.1)
        s["offsets"] = np.concatenate([[0], np.round(share / share[-1] * n)]).astype(np.uint64)
        picks, count = rng.random((nq, labels)).argsort(axis=1)[:, :4], rng.integers(1, 5, nq)
        bit = np.where(np.arange(4) < count[:, None], np.uint64(1) << picks.astype(np.uint64), np.uint64(0))
        s["masks"] = np.bitwise_or.reduce(bit, axis=1)
        s["out"], s["result"] = _outputs(nq, case["k"])
    elif op == "index":
        s["rows"] = _rows(case, seed, n)[0].cpu().numpy()
        s["ts"] = np.arange(n, dtype=np.uint64)
    elif op == "build":
        s["base"] = _rows(case, seed, n)[0]
    elif op == "insert":
        s["base"] = _rows(case, seed, n + case["rows"])[0]
        torch.cuda.synchronize()
        built = _tensor(_graph(s["base"], n, dim, case["degree"], grab.METRIC_L2))
        s["old"] = built.clone()
        s["graph"] = torch.empty(n + case["rows"], case["degree"], dtype=torch.int32, device=DEV)
        s["seed"] = seed
    torch.cuda.synchronize()
    return s


def run(s):
    n, dim, op = s["n"], s["dim"], s["op"]
    if op == "query":
        if s["filter"] == "window":
            return s["idx"].query_range(s["q"], s["k"], 0.1, s["window"][0], s["window"][1])
        if s["filter"] == "bucket":
            return s["idx"].query_local(s["q"], s["k"], s["bucket"])
        return s["idx"].query(s["q"], s["k"])
    if op == "batch":
        return s["idx"].query_range_batch(s["q"], s["k"], s["win"][0], s["win"][1])
    if op == "search":
        grab.search_ex(s["base"].data_ptr(), s["graph"], n, dim, s["degree"], s["q"].data_ptr(), s["nq"], s["k"], s["itopk"], s["width"], 50,
                       s["bitlen"], s["itopk"], s["mask"], d_out=s["out"])
        return s["result"]
    if op == "range":
        q, seeds, (lo, hi) = s["q"].data_ptr(), s["seeds"].data_ptr(), (t.data_ptr() for t in s["ids"])
        out = type("Seeds", (), {"ptr": seeds})
        more = {}
        if s["ordered"]:
            s["layer"].list_grouped(q, s["nq"], 32, 16, 16, d_win_start=s["lo"].data_ptr(), d_win_end=s["hi"].data_ptr(), d_out=out, sync=False,
                                    d_base_ts=s["ts"].data_ptr(), num_base=n, d_id_lo=lo, d_id_hi=hi)
        else:
            s["layer"].list_grouped(q, s["nq"], 32, 16, 16, d_win_start=s["lo"].data_ptr(), d_win_end=s["hi"].data_ptr(), d_out=out, sync=False)
            wrap = [type("Ids", (), {"ptr": p}) for p in (lo, hi)]
            grab.windows_to_id_ranges(s["sorted_ts"].data_ptr(), n, s["lo"].data_ptr(), s["hi"].data_ptr(), s["nq"], wrap[0], wrap[1])
            more = dict(d_rank=s["rank"].data_ptr(), d_graph_rank=s["graph_rank"])
        grab.search_ex(s["base"].data_ptr(), s["graph"], n, dim, s["degree"], q, s["nq"], s["k"], s["itopk"], 4, 50, s["bitlen"], 32, s["mask"],
                       d_seeds=seeds, n_provided=32, filter_kind=grab.FILTER_ID_RANGE, d_win_start=lo, d_win_end=hi,
                       flags=grab.FLAG_FILTER_FIRST, d_out=s["out"], **more)
        return s["result"]
    if op == "window_scan":
        s["scan"].window_topk(s["q"].data_ptr(), s["nq"], s["k"], s["win"][0], s["win"][1], d_out=s["out"])
        return s["result"]
    if op == "bucket_scan":
        s["scan"].bucket_topk(s["offsets"], s["q"].data_ptr(), s["nq"], s["k"], s["masks"], d_out=s["out"])
        return s["result"]
    if op == "index":
        idx = grab.CagraIndex(dim, s["degree"], vmm_max_bytes=4 << 30)
        idx.set_metric(_metric(s))
        idx.add(s["rows"], s["ts"])
        idx.build()
        graph = idx.get_graph()
        idx.close()
        return graph.view(np.int32)
    if op == "build":
        return _tensor(_graph(s["base"], n, dim, s["degree"], _metric(s)))
    # insert: the graph as it was before the batch, then the batch in steps of 64 rows
    base, graph, degree = s["base"], s["graph"], s["degree"]
    graph[:n].copy_(s["old"])
    state = s["seed"]
    for off in range(0, s["rows"], 64):
        m = min(64, s["rows"] - off)
        state = grab.insert(base.data_ptr(), dim, n + off, m, base.data_ptr() + (n + off) * dim * 4, graph.data_ptr(), degree,
                            grab.SearchParams(128, 6, 0, 50, 14), state)
    return graph


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _search_work(n, nq, dim, k, itopk, degree, share):
    """A search that runs to its end expands about every entry of its queue: itopk graph rows, and of their in-filter
    neighbours about 0.4 are rows it has not seen (0.25 to 0.5 by the kernels' own counters; at most the rows there are);
    each row costs dim differences, products and sums.  Rows that several queries read count once."""
    rows = 32 + min(0.4 * itopk * degree * share, 0.5 * n * share)
    read = min(nq * rows, n * share) * 4.0 * dim + min(nq * float(itopk), n * share) * 4.0 * degree
    return {"bytes": read + nq * (4.0 * dim + 12.0 * k), "flops": nq * rows * 3.0 * dim}


def work(case):
    n, dim, op = case["n"], case["dim"], case["op"]
    if op == "query":
        if case["filter"] == "bucket":  # one of twenty buckets holds the rows, and three quarters of a row's slots stay inside it
            return _search_work(n // 20, case["nq"], dim, case["k"], max(case["itopk"], 128), case["degree"] * 3 // 4, 1.0)
        return _search_work(n, case["nq"], dim, case["k"], max(case["itopk"], 64), case["degree"], 0.1 if case["filter"] == "window" else 1.0)
    if op in ("batch", "range"):
        return _search_work(n, case["nq"], dim, case["k"], max(case["itopk"], 64), case["degree"], case["selectivity"])
    if op == "search":
        return _search_work(n, case["nq"], dim, case["k"], case["itopk"], case["degree"], 1.0)
    if op == "window_scan":
        return {"bytes": 4.0 * dim * (n + case["nq"]) + 12.0 * case["nq"] * case["k"], "flops": 2.0 * dim * case["nq"] * case["selectivity"] * n}
    if op == "bucket_scan":
        return {"bytes": 4.0 * dim * (n + case["nq"]) + 12.0 * case["nq"] * case["k"], "flops": 2.0 * dim * case["nq"] * n * 2.5 / case["labels"]}
    if op in ("index", "build"):
        # a distance serves both of its rows: half of all pairs
        return {"bytes": 4.0 * n * (dim + case["degree"]), "flops": float(n) * n * dim}
    w = _search_work(n, case["rows"], dim, 0, 128, case["degree"], 1.0)
    return {"bytes": w["bytes"] + 8.0 * case["rows"] * case["degree"], "flops": w["flops"]}


def tolerance(case):
    """Ids are ids; every distance that comes back is summed in one documented order."""
    return "exact"
