"""The merge at the sizes of its sorts (one wave up to 512 candidates, the
workgroup to 4,096, the select past that), with counts that pack into a word
beside the id and counts too far apart for that, against the oracle."""
import numpy as np
import pytest

from helpers import assert_topk_equal, oracle_search_sample

from genie_amd import Plan, Table
from genie_amd._native import RANGE_DTYPE

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4095, 4096]


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("n", [60_000, 130_000])  # one tile: min(k, matches) candidates; two: up to twice k
def test_merge_sizes(n, far):
    rng = np.random.default_rng(n)
    rows = np.stack([rng.integers(0, 4, n), rng.integers(0, 6, n), rng.integers(0, 300, n)], 1).astype(np.int32)
    q = len(SIZES)
    r = np.zeros(3 * q, RANGE_DTYPE)
    r["query"] = np.repeat(np.arange(q), 3)
    r["dim"] = r["order"] = np.tile(np.arange(3), q)
    r["low"] = [0, 0, 7] * q
    r["up"] = [1, 2, 40] * q
    r["weight"] = [1, 2, 60_000] * q if far else [1, 2, 4] * q
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    k = np.array(SIZES, np.uint32)
    oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), items, n, k, np.arange(q))
    p = Plan(t.device(), q, len(items), 4096, 0, mode=0)
    p.upload(items, q, k)
    p.run()
    ids, cnt = p.download()
    assert_topk_equal(ids, cnt, oi, oc, k, q, f"n={n}")


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("k", [1000, 2048, 4096])
def test_merge_of_more_candidates_than_the_stage(k, far):
    """Six tiles that all hold k objects or more of the least count reached (so
    each emits k): the select, its id bytes skipped, and the selected keys sorted
    packed or, with counts too far apart, as they are."""
    n, q = 6 * 65536 - 17, 3
    rng = np.random.default_rng(k)
    rows = np.stack([np.zeros(n, np.int64), rng.integers(0, 500, n), rng.integers(0, 3000, n)], 1).astype(np.int32)
    r = np.zeros(3 * q, RANGE_DTYPE)
    r["query"] = np.repeat(np.arange(q), 3)
    r["dim"] = r["order"] = np.tile(np.arange(3), q)
    r["low"] = [0, 7, 11] * q
    r["up"] = [0, 7, 11] * q
    r["weight"] = [1, 2, 60_000 if far else 4] * q
    assert 6 * k > 4096
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    kq = np.full(q, k, np.uint32)
    oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), items, n, kq, np.arange(q))
    assert (oc.reshape(q, k)[:, -1] == 1).all()  # the first item's ties
    p = Plan(t.device(), q, len(items), k, 0, mode=0)
    p.upload(items, q, kq)
    for _ in range(2):
        p.run()
        ids, cnt = p.download()
        assert_topk_equal(ids, cnt, oi, oc, k, q, f"k={k}")


def test_merge_few_candidates():
    """k past the matches: padding, and lists of a handful of candidates."""
    n, q = 50_000, 9
    rng = np.random.default_rng(1)
    rows = np.zeros((n, 1), np.int32)
    sizes = [0, 1, 2, 63, 64, 65, 200, 256, 300]
    at = rng.permutation(n)
    o = 0
    for j, s in enumerate(sizes):
        rows[at[o:o + s], 0] = j + 1
        o += s
    r = np.zeros(q, RANGE_DTYPE)
    r["query"] = np.arange(q)
    r["low"] = r["up"] = np.arange(q) + 1
    r["weight"] = 3
    t = Table.from_rows(rows)
    items = t.compile(r, q)
    k = np.full(q, 1000, np.uint32)
    for hash_mode in (0, 1):
        p = Plan(t.device(), q, max(1, len(items)), 1000, 0, mode=0)
        p.set_hash(hash_mode)
        p.upload(items, q, k)
        p.run()
        ids, cnt = p.download()
        oi, oc = oracle_search_sample(t.export()["inv"].view(np.uint32), items, n, k, np.arange(q))
        assert_topk_equal(ids, cnt, oi, oc, k, q, "few")
