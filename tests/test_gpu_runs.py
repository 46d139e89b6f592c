"""Direct-mapped scan over tile-major runs (the plain form's dense select on
indexes with long lists) against the oracle's search of the same work items:
tile edges, items that start and end inside keys, 8- and 16-bit counters,
ties trimmed and tiles with fewer than k matches, set-valued tables, and
compressed tables, whose batches are decoded tile-major (with hash-form
queries in the same batch, also into the posting lists' layout)."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_search_sample, posting_items

import genie_amd
from genie_amd import DIM_DTYPE, Index, Plan, Table, workloads as W

pytestmark = pytest.mark.gpu


def check(table, items, uitems, n, nq, k, where, hash_mode=0, graph=False):
    p = Plan(table.device(), nq, max(1, len(items)), int(np.max(k)), 0, mode=0)
    p.set_hash(hash_mode)
    p.set_sparse(0)
    p.upload(items, nq, k)
    assert not p.sparse_active()
    p.set_graph(graph)
    oi, oc = oracle_search_sample(table.export()["inv"].view(np.uint32), uitems, n, np.broadcast_to(k, (nq,)),
                                  np.arange(nq))
    for _ in range(3 if graph else 1):
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, nq, where)
    return p


def clip(items, rng):
    """Items cut at random positions: they start and end inside keys."""
    out = items.copy()
    span = out["end_pos"] - out["start_pos"]
    out["start_pos"] += (rng.random(len(out)) * span * 0.4).astype(np.int32)
    out["end_pos"] -= (rng.random(len(out)) * span * 0.4).astype(np.int32)
    return out


@pytest.mark.parametrize("n,d,values,radius,wmax,k", [
    (65_535, 9, 300, 6, 1, 50),
    (65_536, 130, 40, 3, 1, 7),      # more items than one window of 64 a query
    (65_537, 12, 700, 40, 1, 3000),  # k above the last tile's objects
    (200_003, 20, 256, 2, 40, 100),  # counts past 255: 16-bit counters
    (131_072, 3, 64, 0, 1, 4096),    # few distinct counts: long ties
    (140_000, 70, 90, 20, 900, 33),  # 16-bit counts in several histogram windows
])
def test_runs_equal_oracle(n, d, values, radius, wmax, k):
    q = 7
    rows = genie_amd.synth.rows(n + d, n, d, genie_amd.synth.ZIPF_PERM, 0.4, 0.0, 0, values - 1, values)
    qv, _ = genie_amd.synth.queries(n + 1, rows, q, noise=radius, lo=0, hi=values - 1)
    w = genie_amd.synth.uniform_int(n + 2, 0, q * d, 1, wmax)
    t = Table.from_rows(rows)
    items = t.compile(W.single_ranges(qv, radius, w), q)
    items = items[items["query"] != 3]  # a query without items
    check(t, items, items, n, q, k, "whole keys", graph=True)
    cut = clip(items, np.random.default_rng(n))
    check(t, cut, cut, n, q, k, "clipped")


@pytest.mark.parametrize("codec", [5, 11, 13])
@pytest.mark.parametrize("n", [65_600, 300_001])
def test_runs_compressed(n, codec):
    d, q = 24, 9
    rows = genie_amd.synth.rows(77, n, d, genie_amd.synth.ZIPF_PERM, 1.1, 0.0, 0, 255, 256)
    qv, _ = genie_amd.synth.queries(78, rows, q, noise=2, lo=0, hi=255)
    r = W.single_ranges(qv, np.where(np.arange(q) < 6, 3, 0).astype(np.int32))
    r = r[(r["query"] < 6) | (r["dim"] == 0)].copy()  # the last three: one exact value each
    rare = np.argsort(np.bincount(rows[:, 0], minlength=256))[100:103]
    r["low"][r["query"] >= 6] = rare
    r["up"][r["query"] >= 6] = rare
    t = Table.from_rows(rows, 1024, True, codec=codec)
    k = np.array([5, 100, 700, 20, 1, 64, 30, 400, 3], np.uint32)
    for merge in (False, True):
        items = t.compile(r, q, merge_runs=merge)
        u = posting_items(t.export(), items)
        p = check(t, items, u, n, q, k, f"codec {codec}", hash_mode=0)
        assert p.decode_active()
        p = check(t, items, u, n, q, k, f"codec {codec} with hash-form queries", hash_mode=-1)
        assert 0 < p.hash_queries() < q
        p.set_sparse(1)  # the posting lists' layout for every query
        p.run()
        a = p.download()
        p.set_sparse(0)
        p.run()
        b = p.download()
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_runs_sets():
    n, q = 90_000, 12
    rp, v = genie_amd.synth.sets(5, n, 3, 30, 300, 0.6)
    qp, qv = genie_amd.synth.sets(6, q, 1, 40, 300, 0.6)
    t = Table.from_sets(rp, v)
    items = t.compile(W.set_ranges(qp, qv, genie_amd.synth.uniform_int(7, 0, len(qv), 1, 9)), q)
    check(t, items, items, n, q, 60, "sets")


@pytest.mark.parametrize("form,q,threads", [("runs", 27_500, 1024), ("lists", 55_500, 512), ("hash", 15_000, 512)])
def test_more_pairs_than_a_launch(form, q, threads):
    """(tile, query) pairs past what one launch takes (2^32 threads), in each
    scan of the plain form; two items of different weights a query."""
    n = 10_000_000
    rows = np.arange(n, dtype=np.int32)[:, None] % 3
    rows[n // 2 + 1::4] = 3
    rows[-4096:] = 4
    first = np.array([np.argmax(rows[:, 0] == v) for v in range(5)])
    t = Table.from_rows(rows)
    v = np.random.default_rng(1).integers(0, 4, (q, 2))
    if form == "hash":  # 3 M postings a query: hash tiles of at most 16,384 objects; the result in the last one
        v[:, 0] %= 3
        v[:, 1] = 4
    r = W.single_ranges(np.concatenate([v[:, :1], v[:, 1:]], 0).astype(np.int32), 0, np.repeat([1, 2], q))
    r["query"] %= q
    r = r[np.argsort(r["query"], kind="stable")]
    items = t.compile(r, q)
    p = Plan(t.device(), q, len(items), 1, 3, mode=0)  # a given bound: not the filter
    p.set_hash(form == "hash")
    p.set_sparse(1 if form == "lists" else 0)
    p.upload(items, q, np.ones(q, np.uint32))
    assert p.hash_queries() == (q if form == "hash" else 0)
    assert -(-n // (16384 if form == "hash" else 65536)) * q * threads > 1 << 32
    p.run()
    ids, cnt = p.download()
    assert p.hash_queries() == (q if form == "hash" else 0)
    same = v[:, 0] == v[:, 1]
    assert np.array_equal(ids, first[v[:, 1]]) and np.array_equal(cnt, np.where(same, 3, 2))


def test_runs_of_more_keys_than_a_launch_of_workgroups():
    """2^24 keys (a workgroup of 256 threads each passed 2^32 threads at index
    creation), most of them without postings."""
    n, K, P = 1000, (1 << 24) + 5, 3_200_000
    rng = np.random.default_rng(2)
    post = rng.integers(0, n, P).astype(np.uint32)
    start = np.zeros(K + 1, np.uint64)
    ends = np.sort(rng.choice(K - 1, P, replace=False)) + 1  # a key of one posting before each
    start[ends] = 1
    start[K] = 1
    start = np.minimum(np.cumsum(start), P).astype(np.uint64)
    ix = Index.create(n, 1, post, start, np.zeros(K, np.uint32), np.array([0, P], np.uint32), single_value=False)
    q, k = 3, 50
    items = np.zeros(q, DIM_DTYPE)
    items["query"] = np.arange(q)
    items["start_pos"] = [0, 100_000, P - 700_000]
    items["end_pos"] = [500_000, P, P]
    items["weight"] = 1
    oi, oc = oracle_search_sample(post, items, n, np.full(q, k), np.arange(q))
    p = Plan(ix, q, q, k, 65535, mode=0)
    p.set_hash(0)
    p.set_sparse(0)
    p.upload(items, q, np.full(q, k, np.uint32))
    p.run()
    ids, cnt = p.download()
    assert_topk_equal(ids, cnt, oi, oc, k, q, "keys")
