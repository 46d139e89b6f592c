"""Sample histograms with shifted bins (weighted dense batches, set batches):
a query whose k passes its matches counting at least one bin's width still
gets the objects that count less than that."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_topk_batch
from oracle import oracle as O

import genie_amd
from genie_amd import Plan, Table, workloads as W

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
