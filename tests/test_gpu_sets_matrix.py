"""Set form on the matrix cores (hot keys as a product, mid keys scattered from
tile-major windows, tail keys from postings sorted by tile) against the
oracle's search of the same items: tile edges, byte and 16-bit counters,
repeated tokens, multiplicities an i8 does not hold, keys of one class only,
partial groups, compressed tables, graph replays."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_search_sample, posting_items

import genie_amd
from genie_amd import Index, Plan, Table, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,q,vocab,skew,wmax,k", [
    (2047, 33, 200, 1.05, 1, 10),        # one tile, one object short of it; a group of one query
    (2048, 5, 3000, 1.05, 3, 2048),      # k = every object
    (2049, 32, 60, 0.5, 2, 100),         # every key hot
    (70_001, 70, 40_000, 1.05, 4, 50),   # hot, mid and tail keys
    (70_001, 40, 40_000, 1.05, 60, 50),  # 16-bit counters
    (30_000, 100, 30_000, 0.0, 1, 20),   # a flat vocabulary: short runs, many ties
    (40_001, 64, 1500, 0.0, 1, 30),      # ties that half fill a tile's stage
])
@pytest.mark.parametrize("codec", [0, 11])
def test_matrix_form_equals_oracle(n, q, vocab, skew, wmax, k, codec):
    rp, v = genie_amd.synth.sets(n, n, 3, 30, vocab, skew)
    qp, qv = genie_amd.synth.sets(n + 1, q, 1, 40, vocab, skew)
    w = genie_amd.synth.uniform_int(n + 2, 0, len(qv), 1, wmax)
    if wmax > 50:  # a token named twice may not pass the largest weight per key
        _, first = np.unique(np.repeat(np.arange(q), np.diff(qp)) * vocab + qv, return_index=True)
        keep = np.zeros(len(qv), bool)
        keep[first] = True
        cnt = np.add.reduceat(keep.astype(np.int64), qp[:-1])
        qp, qv, w = np.concatenate([[0], np.cumsum(cnt)]), qv[keep], w[keep]
    t = Table.from_sets(rp, v, **(dict(max_length=1024, load_balance=True, codec=codec) if codec else {}))
    check(t, W.set_ranges(qp, qv, w), n, q, k, codec)


def test_matrix_form_multiplicities():
    """The most frequent token 200 times in some documents: not an i8 column."""
    rng = np.random.default_rng(3)
    docs = [np.sort(rng.integers(0, 500, rng.integers(3, 20))) for _ in range(5000)]
    for i in range(0, 5000, 97):
        docs[i] = np.concatenate([np.full(200, 7), docs[i]])
    rp = np.concatenate([[0], np.cumsum([len(x) for x in docs])]).astype(np.int64)
    t = Table.from_sets(rp, np.concatenate(docs).astype(np.int32))
    q = 20
    qv = [np.unique(np.append(rng.integers(0, 500, 15), 7 if j % 2 else 3)) for j in range(q)]
    qp = np.concatenate([[0], np.cumsum([len(x) for x in qv])])
    flat = np.concatenate(qv).astype(np.int32)
    check(t, W.set_ranges(qp, flat, rng.integers(1, 9, len(flat))), 5000, q, 30, 0)


@pytest.mark.parametrize("weights", [
    [63, 63, 1], [32] * 4, [50, 50, 50, 30], [60, 60, 60], [51] * 5,  # bounds 127, 128, 180, 180, 255 of byte counters
    [51] * 5 + [1],                                                   # 256: 16-bit counters
    [1] * 130, [1] * 250, [2] * 125 + [1] * 5,
])
@pytest.mark.parametrize("holders", [4, 40])  # tail keys, mid keys
def test_matrix_form_scattered_counts_past_127(weights, holders):
    """Documents that hold every token of a query besides the most frequent
    ones, at each place in a counter word, at both ends of a tile and as the
    index's last object, beside documents that hold one of them or none; k past
    the matches."""
    n, m = 20_003, len(weights)
    rng = np.random.default_rng(m)
    docs = [np.sort(rng.choice(64, 2, replace=False)) for _ in range(n)]  # the 64 longest lists
    at = np.concatenate([[0, 2047, 2049, n - 1], 4100 + 5 * rng.choice(3000, holders - 4, replace=False)])
    for i, o in enumerate(at):
        docs[o] = np.append(docs[o], 1000 + np.arange(m))
        if i % 2 and o + 1 < n:  # a neighbour with a count of its own
            docs[o + 1] = np.append(docs[o + 1], 1000 + i % m)
    rp = np.concatenate([[0], np.cumsum([len(x) for x in docs])]).astype(np.int64)
    t = Table.from_sets(rp, np.concatenate(docs).astype(np.int32))
    assert {int(o) % 4 for o in at} >= {0, 1, 2, 3}
    q = 3  # every token; all but one; every token and a frequent one
    qv = [1000 + np.arange(m), 1000 + np.arange(1, m), np.append(5, 1000 + np.arange(m))]
    wv = [weights, weights[1:], [3] + list(weights)]
    qp = np.concatenate([[0], np.cumsum([len(x) for x in qv])])
    check(t, W.set_ranges(qp, np.concatenate(qv).astype(np.int32), np.concatenate(wv).astype(np.int32)), n, q, 200, 0)


def test_matrix_form_of_unordered_postings():
    """A compressed table whose posting array, beside the words, lists every
    key's objects in descending order: the matrix form is built from the words."""
    n, q, k = 30_000, 40, 50
    rp, v = genie_amd.synth.sets(5, n, 3, 30, 20_000, 1.05)
    docs = [np.unique(v[rp[i]:rp[i + 1]]) for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(x) for x in docs])]).astype(np.int64)
    t = Table.from_sets(rp, np.concatenate(docs).astype(np.int32), max_length=1024, load_balance=True, codec=11)
    e = t.export()
    start = np.concatenate([[0], e["inv_pos"][e["keyseg"][1:]]]).astype(np.int64)
    post = e["inv"].copy()
    for a, b in zip(start[:-1], start[1:]):
        post[a:b] = post[a:b][::-1]
    ix = Index.create(n, 1, post, start, np.zeros(len(start) - 1, np.uint32), e["inv_pos"], False, 11, e["words"],
                      e["cpos"])
    qp, qv = genie_amd.synth.sets(6, q, 1, 40, 20_000, 1.05)
    items = t.compile(W.set_ranges(qp, qv, np.full(len(qv), 2)), q, merge_runs=True)
    oi, oc = oracle_search_sample(e["inv"].view(np.uint32), posting_items(e, items), n, np.full(q, k), np.arange(q))
    p = Plan(ix, q, len(items), k, 0, mode=2)
    p.upload(items, q, np.full(q, k, np.uint32))
    assert p.form() == "set"
    p.run()
    ids, cnt = p.download()
    assert_topk_equal(ids, cnt, oi, oc, k, q, "unordered")


def test_forms_of_successive_batches():
    """Batches for the matrix form and for the forward lists in turn through one
    plan (the slots of a batch of long runs end its gathering before its last
    group), and a group of more keys than the lists' table holds."""
    n, k = 150_000, 20
    rp, v = genie_amd.synth.sets(8, n, 3, 12, 4000, 0.0)
    v = np.where(np.arange(len(v)) % 3 > 0, v % 130, v).astype(np.int32)  # 130 tokens of long runs
    t = Table.from_sets(rp, v)
    rng = np.random.default_rng(4)
    few = [rng.choice(np.arange(130, 4000), 5, replace=False) for _ in range(100)]
    many = [rng.choice(130, 100, replace=False) for _ in range(70)]
    last = [rng.choice(np.arange(130, 4000), 3, replace=False) for _ in range(32)] + many[:64]
    wide = [np.arange(200 * (j % 19), 200 * (j % 19) + 200) for j in range(40)]  # 3,800 keys in 32 queries
    p = Plan(t.device(), 100, 20_000, k, 0, mode=2)
    for qs, form in ((few, "set"), (many, "set"), (few, "set"), (last, "set"), (wide, "plain"), (few, "set")):
        q, qp = len(qs), np.concatenate([[0], np.cumsum([len(x) for x in qs])])
        items = t.compile(W.set_ranges(qp, np.concatenate(qs).astype(np.int32), np.full(int(qp[-1]), 3)), q)
        oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), items, n, np.full(q, k), np.arange(q))
        p.upload(items, q, np.full(q, k, np.uint32))
        assert p.form() == form
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, q, form)


def test_matrix_form_keeps_a_compressed_index_small():
    rp, v = genie_amd.synth.sets(5, 70_001, 3, 30, 40_000, 1.05)
    plain = Table.from_sets(rp, v)
    comp = Table.from_sets(rp, v, max_length=1024, load_balance=True, codec=11)
    assert comp.device().bytes() < plain.device().bytes()


def check(t, ranges, n, q, k, codec):
    items = t.compile(ranges, q, merge_runs=bool(codec))
    export = t.export()
    u = posting_items(export, items) if codec else items
    oi, oc = oracle_search_sample(export["inv"].view(np.uint32), u, n, np.full(q, k), np.arange(q))
    p = Plan(t.device(), q, len(items), k, 0, mode=2)
    p.upload(items, q, np.full(q, k, np.uint32))
    assert p.form() == "set"
    p.set_graph(True)
    for _ in range(3):
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, q, f"n={n}")
