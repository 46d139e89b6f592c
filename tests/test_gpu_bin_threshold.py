"""Sample histograms with shifted bins (weighted dense batches, set batches):
a query whose k passes its matches counting at least one bin's width still
gets the objects that count less than that, without room for every object."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_search_sample, oracle_topk_batch
from oracle import oracle as O

import genie_amd
from genie_amd import Plan, Table, mem_info, workloads as W

pytestmark = pytest.mark.gpu


def test_weighted_dense_small_counts():
    n, d, k = 3000, 64, 2900
    rows = genie_amd.synth.rows(9, n, d, genie_amd.synth.UNIFORM, 0.0, 0.0, 0, 7, 8)
    r = W.single_ranges(rows[:2], 2)
    r = r[(r["query"] == 0) | (r["dim"] < 3)].copy()
    r["weight"] = np.where(r["dim"] == 0, 9.0, 1.0)  # query 1: counts 1, 2, 9, 10, 11; bins of 4
    t = Table.from_rows(rows)
    items = t.compile(r, 2)
    p = Plan(t.device(), 2, len(items), k, 0, mode=2)
    p.upload(items, 2, np.full(2, k, np.uint32))
    assert p.form() == "dense"
    p.run()
    ids, cnt = p.download()
    ri, rc = oracle_topk_batch(lambda q: O.count_exhaustive_single(rows, r[r["query"] == q]), 2, k)
    assert_topk_equal(ids, cnt, ri, rc, k, 2, "small counts")


@pytest.mark.parametrize("lists", [False, True])
def test_few_matches_take_little_room(lists):
    """Weighted queries with fewer matches than k, of counts below a bin's
    width among others: room for their matches, not for queries x objects.
    `lists`: a flat vocabulary of long lists, which stays on the forward
    lists."""
    n, q, k = 300_000, 1024, 50
    rp, v = genie_amd.synth.sets(3, n, 2, 16 if lists else 20, 300 if lists else 400_000, 0.0)
    if lists:  # rare tokens, for the queries
        v = v.copy()
        at = np.random.default_rng(1).choice(len(v), 4000, replace=False)
        v[at] = 300 + np.arange(4000) % 400
    rng = np.random.default_rng(2)
    qv = np.array([rng.choice(400 if lists else 400_000, 3, replace=False) for _ in range(q)]).astype(np.int32)
    qv += 300 if lists else 0
    if lists:  # long queries in every group
        wide = np.arange(0, q, 32)
        rest = {int(j): np.arange(300, dtype=np.int32) for j in wide}
    qs = [np.concatenate([qv[j], rest[j]]) if lists and j in rest else qv[j] for j in range(q)]
    qp = np.concatenate([[0], np.cumsum([len(x) for x in qs])])
    w = genie_amd.synth.uniform_int(4, 0, int(qp[-1]), 1, 50)
    t = Table.from_sets(rp, v)
    items = t.compile(W.set_ranges(qp, np.concatenate(qs), w), q)
    ix = t.device()
    free = mem_info()[0]
    p = Plan(ix, q, len(items), k, 0, mode=2)
    p.upload(items, q, np.full(q, k, np.uint32))
    assert p.form() == "set"
    p.run()
    ids, cnt = p.download()
    used = free - mem_info()[0]
    oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), items, n, np.full(q, k), np.arange(q))
    assert_topk_equal(ids, cnt, oi, oc, k, q, "few")
    assert used < 500e6, used
