"""Filter form of selective single-key, one-weight queries (objects of several
postings by a bit filter, the rest from the heads of the lists) against the
oracle's search: k past the objects of several postings, one list only, a
weight above 1, tile counts, short lists without directory rows, empty
queries, crowded low ids, repeated ids in set-valued lists."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_search_sample, posting_items

import genie_amd
from genie_amd import Plan, Table, workloads as W

pytestmark = pytest.mark.gpu


def check(t, items, u, n, q, k, hashed=None):
    oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), u, n, np.broadcast_to(k, (q,)), np.arange(q))
    kq = np.ascontiguousarray(np.broadcast_to(np.asarray(k, np.uint32), (q,)))
    p = Plan(t.device(), q, max(1, len(items)), int(kq.max()), 0, mode=0)
    p.upload(items, q, kq)
    if hashed is not None:
        assert p.hash_queries() == hashed
    p.set_graph(True)
    for _ in range(3):
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, q, f"n={n}")
    return p


@pytest.mark.parametrize("n,d,buckets,k,weight", [
    (100_000, 40, 900, 20, 1),     # one tile, lists of about 111 (no directory rows)
    (300_000, 24, 512, 1024, 3),   # most of the result are objects of one posting
    (600_001, 120, 2048, 60, 1),   # three tiles of 293-id lists
    (400_000, 1, 4096, 200, 2),    # one list: k past its length
    (2_000_003, 64, 1100, 100, 1), # eight tiles
])
@pytest.mark.parametrize("codec", [0, 13])
def test_filter_equals_oracle(n, d, buckets, k, weight, codec):
    q = 9
    rows = genie_amd.synth.rows(n, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, buckets - 1, buckets)
    qv, _ = genie_amd.synth.queries(n + 1, rows, q, redraw_p=0.5, n_values=buckets)
    r = W.single_ranges(qv, 0, np.full(q * d, weight))
    r = r[(r["query"] != 4) & ((r["query"] != 6) | (r["dim"] == 0))]  # 4 empty, 6 a single list
    t = Table.from_rows(rows, **(dict(max_length=1024, load_balance=True, codec=codec) if codec else {}))
    items = t.compile(r, q, merge_runs=bool(codec))
    check(t, items, posting_items(t.export(), items) if codec else items, n, q, k)


def test_filter_crowded_low_ids():
    """Every matching object lies at the start of the index: the first bound of
    the fill holds far more ids than it aims at."""
    n, d, q = 600_000, 6, 5
    rows = genie_amd.synth.rows(3, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 3999, 4000)
    rows[:9000] = 4000 + np.arange(9000)[:, None] // 1500 + np.zeros(d, np.int32)
    r = W.single_ranges(np.tile(np.arange(4000, 4000 + q)[:, None], (1, d)).astype(np.int32), 0)
    r = r[(r["dim"] == 0) | (r["query"] > 2)]
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    check(t, items, items, n, q, 300)


@pytest.mark.parametrize("at", [0, 300_000])
def test_fill_among_crowded_ids(at):
    """Objects of one posting only, all within 9,000 ids: more of them below the
    fill's first bound than its table takes, though few are needed."""
    n, d, q = 600_000, 6, 3
    rows = genie_amd.synth.rows(3, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 3999, 4000)
    for j in range(d):
        rows[at + 1500 * j:at + 1500 * j + 1500, j] = 5000
    r = W.single_ranges(np.full((q, d), 5000, np.int32), 0)
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    p = check(t, items, items, n, q, 300, q)
    assert p.hash_queries() == q  # none was given to the direct kernels


@pytest.mark.parametrize("n,shared,span,k", [
    (2_000_000, 9000, 900_000, 60),       # two tiles, every id in the first: its table fills up
    (2_000_000, 9000, 900_000, 1024),
    (4_000_000, 16_200, 1_900_000, 700),  # two tiles, more bits set than a tile's share
    (2_000_000, 8100, 900_000, 60),       # nearly full
])
def test_filter_tiles_of_many_shared_objects(n, shared, span, k):
    """Objects that share two or three of a query's values, more of them in a
    tile than the table of the filter takes: counted in quarters."""
    d, q = 8, 6
    rng = np.random.default_rng(shared)
    rows = genie_amd.synth.rows(3, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 3999, 4000)
    at = rng.choice(span, shared, replace=False)
    i = np.arange(shared)
    for e in (0, 1):
        rows[at, (i + e) % d] = 5000
    rows[at[::50], (i[::50] + 2) % d] = 5000
    r = W.single_ranges(np.full((q, d), 5000, np.int32), 0, np.full(q * d, 2))
    r = r[(r["query"] != 1) | (r["dim"] < 6)]
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    p = check(t, items, items, n, q, k, q)
    assert p.hash_queries() == q  # none was given to the direct kernels


def test_filter_sets():
    n, q = 500_000, 20
    rp, v = genie_amd.synth.sets(5, n, 3, 30, 3000, 0.2)
    qp, qv = genie_amd.synth.sets(6, q, 1, 6, 3000, 0.2)
    t = Table.from_sets(rp, v)
    items = t.compile(W.set_ranges(qp, qv, np.full(len(qv), 2)), q)
    check(t, items, items, n, q, 90)


@pytest.mark.parametrize("mode", [0, 2])
def test_batch_without_items(mode):
    rows = genie_amd.synth.rows(3, 50_000, 4, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 3999, 4000)
    t = Table.from_rows(rows)
    p = Plan(t.device(), 3, 1, 20, 0, mode=mode)
    p.upload(np.zeros(0, genie_amd.DIM_DTYPE), 3, np.full(3, 20, np.uint32))
    p.run()
    ids, cnt = p.download()
    assert not ids.any() and not cnt.any()


@pytest.mark.parametrize("q", [21, 701])  # few filter tiles: the hash kernel takes them; many: both kernels
@pytest.mark.parametrize("codec", [0, 13])
def test_filter_and_hash_queries_in_one_batch(q, codec):
    n, d = 1_000_000, 36
    rows = genie_amd.synth.rows(11, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 1499, 1500)
    qv, _ = genie_amd.synth.queries(12, rows, q, redraw_p=0.4, n_values=1500)
    w = np.ones((q, d), np.int64)
    w[::2, 3] = 2  # every second query: two weights
    t = Table.from_rows(rows, **(dict(max_length=1024, load_balance=True, codec=codec) if codec else {}))
    items = t.compile(W.single_ranges(qv, 0, w.reshape(-1)), q, merge_runs=bool(codec))
    check(t, items, posting_items(t.export(), items) if codec else items, n, q, 30, q)


@pytest.mark.parametrize("kind", ["filter", "compressed", "sets"])
def test_batches_without_room_for_a_form(kind):
    """A plan that may not take a form's buffers runs the form without them, in
    turn with batches that may."""
    n, q, k = 400_000, 60, 40
    codec = dict(max_length=1024, load_balance=True, codec=11) if kind != "filter" else {}
    if kind == "sets":
        n = 60_000
        rp, v = genie_amd.synth.sets(5, n, 3, 30, 40_000, 1.0)
        qp, qv = genie_amd.synth.sets(6, q, 1, 30, 40_000, 1.0)
        t, r = Table.from_sets(rp, v, **codec), W.set_ranges(qp, qv, np.full(len(qv), 2))
    else:
        rows = genie_amd.synth.rows(7, n, 40, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 1999, 2000)
        t, r = Table.from_rows(rows, **codec), W.single_ranges(rows[:q], 0)
    items = t.compile(r, q, merge_runs=bool(codec))
    u = posting_items(t.export(), items) if codec else items
    oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), u, n, np.full(q, k), np.arange(q))
    p = Plan(t.device(), q, len(items), k, 0, mode=2 if kind == "sets" else 0)
    for limit in (0, 1, 0, 1):
        p.set_scratch(limit)
        p.upload(items, q, np.full(q, k, np.uint32))
        if kind == "sets":
            assert p.form() == "set"
        else:
            assert p.hash_queries() == q
            assert p.decode_active() == (kind == "compressed" and limit == 0)
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, q, f"{kind} {limit}")
