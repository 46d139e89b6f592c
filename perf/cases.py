"""What a user of this framework has it do: the calls that the speed of the
match-count top-k search is judged by.

A case is a dict of plain values:
  data      "ranks"    rows of 8-bit feature values, each dim a permutation of Zipf(1.1) ranks
            "normal"   rows of clamped normal values (SIFT-like), `values` of them per dim
            "buckets"  rows of LSH buckets, uniform over `values`
            "sets"     documents of `len_lo`..`len_hi` tokens, Zipf(1.05) over `values`
  n, d      objects and dims (documents, 1)
  q, k      queries of a batch and results per query ("mixed": 10, 100 or 1000 by query)
  radius    a query's range around its value in every dim (-1: 0, 2 or 5 by query)
  weight    largest query weight (weights are uniform over 1..weight)
  codec     COMPRESSION_TYPE of the index (0: uncompressed posting lists)
  mode      the plan's mode: 2 automatic, 0 plain (one query per workgroup)
  call      "resident"  a plan holds the uploaded batch in HBM; the results stay in HBM too
            "upload"    a new batch through a kept plan: upload, run, results to the host
            "once"      the one-call search, host arrays in and out
            "server"    a backlog of single requests through the serving loop
"""
import ctypes

import numpy as np
import torch

import genie_amd
from genie_amd import DIM_DTYPE, Plan, Server, Table, match_topk, synth
from genie_amd import workloads as W

_c = ctypes.CDLL(genie_amd.lib_paths()[0])
_c.genie_hip_plan_download.argtypes = [ctypes.c_void_p] * 4
_c.genie_hip_plan_download.restype = ctypes.c_int

MIXED_K = np.array([10, 100, 1000], np.uint32)


def _case(name, data, n, d, q, k, *, values=256, radius=0, weight=1, codec=0, mode=2, call="resident", len_lo=0,
          len_hi=0):
    c = dict(data=data, n=n, d=d, q=q, k=k, values=values, radius=radius, weight=weight, codec=codec, mode=mode,
             call=call, len_lo=len_lo, len_hi=len_hi)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the examples' size: a thousand SIFT descriptors, a hundred exact-match queries, one call
        _case("sift_1k_once", "normal", 1000, 128, 100, 10, call="once"),
        # one interactive query at a time over a million rows, through a plan that the program keeps
        _case("one_query_1m", "ranks", 1_000_000, 128, 1, 10, radius=2, call="upload"),
        # the headline benchmark: a batch of range queries over a million rows
        _case("batch_1m_128", "ranks", 1_000_000, 128, 1024, 100, radius=2),
        # the same with query weights
        _case("batch_weighted", "ranks", 500_000, 96, 512, 100, radius=2, weight=4),
        # sizes that fit no tile, wide ranges, long result lists
        _case("batch_ragged_k1000", "ranks", 300_007, 77, 333, 1000, radius=5),
        # the reference's own path: posting lists of a compressed index, one query per workgroup
        _case("plain_compressed", "ranks", 600_000, 64, 256, 100, radius=2, codec=11, mode=0),
        # features of more than 256 values per dim: long ranges, many keys per item
        _case("wide_values", "normal", 400_000, 48, 384, 100, values=2048, radius=40),
        # approximate nearest neighbours: LSH buckets, exact match, selective lists
        _case("lsh_4m", "buckets", 4_000_000, 64, 4096, 100, values=8192),
        # a smaller LSH index kept compressed
        _case("lsh_compressed", "buckets", 1_000_000, 48, 1500, 50, values=4096, codec=13),
        # document search: token sets, weighted queries, mixed k
        _case("sets_2m", "sets", 2_000_000, 1, 16384, "mixed", values=1_000_000, weight=4, len_lo=5, len_hi=40),
        # tweets: short documents, small batches of queries over them
        _case("sets_small", "sets", 150_000, 1, 200, 20, values=50_000, weight=1, len_lo=3, len_hi=25),
        # the serving loop catching up with a backlog of mixed requests over a compressed index
        _case("serving_backlog", "ranks", 500_000, 128, 1024, "mixed", radius=-1, codec=11, call="server"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["batch", "batch", "plain", "wide", "lsh", "lsh", "sets", "sets", "server"])
    if kind == "batch":  # the dense batches and the single calls
        call = rng.choice(["resident", "resident", "upload", "once"])
        return _case(None, rng.choice(["ranks", "normal"]), _log(rng, 1000, 1_000_000), rng.randint(3, 128),
                     _log(rng, 1, 1024 if call == "resident" else 128), _log(rng, 1, 1000), radius=rng.randint(0, 6),
                     weight=rng.choice([1, 1, 1, 3, 4, 9]), codec=rng.choice([0, 0, 11]), call=call)
    if kind == "plain":
        return _case(None, "ranks", _log(rng, 20_000, 600_000), rng.randint(8, 96), _log(rng, 4, 256),
                     _log(rng, 1, 1000), radius=rng.randint(0, 3), weight=rng.choice([1, 1, 5]),
                     codec=rng.choice([0, 5, 11, 13]), mode=0)
    if kind == "wide":
        v = rng.choice([300, 512, 1000, 2048, 4096])
        return _case(None, "normal", _log(rng, 40_000, 400_000), rng.randint(8, 64), _log(rng, 4, 384),
                     _log(rng, 1, 500), values=v, radius=rng.randint(v // 200, v // 40), weight=rng.choice([1, 1, 3]))
    if kind == "lsh":
        return _case(None, "buckets", _log(rng, 200_000, 4_000_000), rng.randint(12, 64), _log(rng, 8, 4096),
                     _log(rng, 5, 500), values=rng.choice([1024, 2048, 4096, 8192]), codec=rng.choice([0, 0, 13]))
    if kind == "sets":
        n = _log(rng, 20_000, 2_000_000)
        return _case(None, "sets", n, 1, min(_log(rng, 16, 16384), 3 * 10**10 // n),
                     rng.choice([10, 33, 100, 700, "mixed"]), values=_log(rng, 5000, 1_000_000),
                     weight=rng.choice([1, 2, 4, 7]), len_lo=rng.randint(1, 8), len_hi=rng.randint(9, 40))
    return _case(None, "ranks", _log(rng, 50_000, 500_000), rng.randint(32, 128), _log(rng, 64, 1024),
                 "mixed", radius=-1, codec=rng.choice([0, 11]), call="server")


def _inputs(case, seed):
    """The data on the host and the queries on it: (table data, ranges, k per query)."""
    s = 1000 * int(seed) + 17
    n, d, q, V = case["n"], case["d"], case["q"], case["values"]
    if case["k"] == "mixed":  # a third of each, in random order
        k = MIXED_K[np.random.default_rng(s + 3).permutation(q) % 3]
    else:
        k = np.full(q, case["k"], np.uint32)
    if case["data"] == "sets":
        row_ptr, vals = synth.sets(s, n, case["len_lo"], case["len_hi"], V, 1.05)
        q_ptr, q_vals = synth.sets(s + 1, q, 1, 64, V, 1.05)
        w = synth.uniform_int(s + 2, 0, len(q_vals), 1, case["weight"])
        return (row_ptr, vals), W.set_ranges(q_ptr, q_vals, w), k
    if case["data"] == "buckets":
        rows = synth.rows(s, n, d, synth.UNIFORM, 0.0, 0.0, 0, V - 1, V)
        qv, _ = synth.queries(s + 1, rows, q, redraw_p=0.3, n_values=V)
    elif case["data"] == "normal":
        rows = synth.rows(s, n, d, synth.NORMAL, 100.0 * V / 256, 40.0 * V / 256, 0, V - 1)
        qv, _ = synth.queries(s + 1, rows, q, noise=3 * V // 256, lo=0, hi=V - 1)
    else:
        rows = synth.rows(s, n, d, synth.ZIPF_PERM, 1.1, 0.0, 0, V - 1, V)
        qv, _ = synth.queries(s + 1, rows, q, noise=3, lo=0, hi=V - 1)
    radius = case["radius"]
    if radius < 0:
        radius = np.array([0, 2, 5], np.int32)[synth.uniform_int(s + 4, 0, q, 0, 2)]
    w = None if case["weight"] == 1 else synth.uniform_int(s + 2, 0, q * d, 1, case["weight"])
    return rows, W.single_ranges(qv, radius, w), k


def prepare(case, seed):
    data, ranges, k = _inputs(case, seed)
    q, codec = case["q"], case["codec"]
    seg = dict(max_length=1024, load_balance=True, codec=codec) if codec else {}
    if case["data"] == "sets":
        table = Table.from_sets(data[0], data[1], **seg)
    else:
        table = Table.from_rows(data, **seg)
    index = table.device()
    # requests of a compressed table: the consecutive segments of a range as one item
    items = table.compile(ranges, q, merge_runs=bool(codec))
    st = dict(case=case, table=table, index=index, items=items, k=k, call=case["call"])
    if case["call"] == "server":
        st["server"] = Server(index, executors=4, max_batch=256, max_k=1000, mode=case["mode"])
        st["ptr"] = np.searchsorted(items["query"], np.arange(q + 1)).astype(np.uint64)
        st["arrival"] = np.zeros(q)
    elif case["call"] != "once":
        st["plan"] = Plan(index, q, len(items), int(k.max()), 0, mode=case["mode"])
        if case["call"] == "resident":
            st["plan"].upload(items, q, k)
            st["ids"] = torch.zeros(int(k.sum()), dtype=torch.int32, device="cuda")
            st["counts"] = torch.zeros(int(k.sum()), dtype=torch.int32, device="cuda")
    return st


def run(st):
    call = st["call"]
    if call == "once":
        ids, counts = match_topk(st["index"], st["items"], st["case"]["q"], st["k"])
    elif call == "upload":
        p = st["plan"]
        p.upload(st["items"], st["case"]["q"], st["k"])
        p.run()
        ids, counts = p.download()
    elif call == "server":
        _, ids, counts, _ = st["server"].replay(st["items"], st["ptr"], st["k"], st["arrival"])
    else:
        p, ids, counts = st["plan"], st["ids"], st["counts"]
        p.run()
        if _c.genie_hip_plan_download(p.handle, None, ids.data_ptr(), counts.data_ptr()):
            raise RuntimeError("download")
    return dict(ids=ids, counts=counts)


def _hit(case):
    """Share of a dim's objects that one range matches, about."""
    if case["data"] == "normal":
        return min(1.0, (2 * max(case["radius"], 0) + 1) / (2.5 * 40.0 * case["values"] / 256))
    r = 2 if case["radius"] < 0 else case["radius"]
    return min(1.0, (2 * r + 1) / case["values"])


def work(case):
    """Bytes: every (object, dim) value that the batch's ranges can match, read once in the smallest whole number of
    bytes that holds it (a posting of 4 bytes where lists are so selective that reading only them is less; 4 bytes a
    token); the work items and k once; ids and counts once.  Operations: one addition per matched posting."""
    n, d, q = case["n"], case["d"], case["q"]
    ktot = q * (370 if case["k"] == "mixed" else case["k"])
    if case["data"] == "sets":
        occ = n * (case["len_lo"] + case["len_hi"]) / 2
        items = q * 32.5
        V = case["values"]
        p = np.arange(1, V + 1, dtype=np.float64) ** -1.05
        p /= p.sum()
        flops = occ * items * float((p * p).sum())  # tokens of a query and a document that are the same
        data = 4.0 * occ
    else:
        items = q * d
        flops = float(n) * d * q * _hit(case)
        code = 1 if case["values"] <= 256 else 2
        data = min(float(n) * d * code, 4.0 * flops)
    return {"bytes": int(data + items * DIM_DTYPE.itemsize + 4 * q + 8 * ktot), "flops": int(flops)}


def tolerance(case):
    return "exact"  # counts are integers, and equal counts are ordered by id


def _top(counts, kk):
    """ids, counts of the k largest of each row, ties by id; objects that count nothing are (0, 0)."""
    n = counts.shape[1]
    low = torch.arange(n, device=counts.device, dtype=torch.int64)
    key = (counts.to(torch.int64) << 32) + ((1 << 32) - 1 - low)
    out_i, out_c = [], []
    m = min(n, int(max(kk)))
    best = torch.topk(key, m, dim=1, sorted=True).values
    for r, k in enumerate(kk):
        b = best[r, :int(k)]
        c = b >> 32
        i = torch.where(c > 0, (1 << 32) - 1 - (b & 0xFFFFFFFF), torch.zeros_like(b))
        pad = int(k) - b.numel()
        if pad > 0:
            c, i = (torch.cat([x, x.new_zeros(pad)]) for x in (c, i))
        out_i.append(i)
        out_c.append(c)
    return torch.cat(out_i), torch.cat(out_c)


def exact(case, seed):
    n, q, d = case["n"], case["q"], case["d"]
    if case["data"] == "sets" and float(n) * q > 2e9:
        return None
    data, ranges, k = _inputs(case, seed)
    ids, cnt = [], []
    if case["data"] == "sets":
        row_ptr, vals = data
        vals = torch.from_numpy(vals).cuda().long()
        obj = torch.repeat_interleave(torch.arange(n, device="cuda"), torch.from_numpy(np.diff(row_ptr)).cuda())
        qs, tok = torch.from_numpy(ranges["query"].copy()).cuda().long(), torch.from_numpy(ranges["low"].copy()).cuda().long()
        wt = torch.from_numpy(ranges["weight"].copy()).cuda().long()
        for j in range(q):
            w = torch.zeros(case["values"] + 1, dtype=torch.int64, device="cuda")
            mine = qs == j
            w.index_add_(0, tok[mine], wt[mine])
            c = torch.zeros(n, dtype=torch.int64, device="cuda").index_add_(0, obj, w[vals])
            i, c = _top(c[None], k[j:j + 1])
            ids.append(i)
            cnt.append(c)
    else:
        cols = torch.from_numpy(data).cuda().t().contiguous().to(torch.int16)
        lo, hi, wt = (torch.from_numpy(ranges[f].astype(np.int32)).cuda().view(q, d) for f in ("low", "up", "weight"))
        step = max(1, min(32, 2**26 // n))
        for j in range(0, q, step):
            c = torch.zeros((min(step, q - j), n), dtype=torch.int32, device="cuda")
            for x in range(d):
                v = cols[x]
                hit = (v >= lo[j:j + step, x, None]) & (v <= hi[j:j + step, x, None])
                c += hit * wt[j:j + step, x, None]
            i, c = _top(c, k[j:j + step])
            ids.append(i)
            cnt.append(c)
    return dict(ids=torch.cat(ids), counts=torch.cat(cnt))
