"""The flat scan on the 16-bit matrix unit, at the sizes where its split of the work changes: row
widths around its 16-dim steps (8-dim padding included), batches around its 128-, 256- and 512-query
blocks, row counts around its 16-row groups and 64-row tiles, list lengths (k 10/11, 21/22, 43),
magnitudes far from 1, and for rows wider than 128 dims around the 32-dim chunks, 256-row tiles and
64- and 256-query blocks. Distances must equal the oracle's bit for bit and labels must agree within
equal-distance groups, so no tolerance is involved."""

import numpy as np
import pytest

import quiver_amd as quiver
from oracle.oracle import rows_bitmap
from parity import assert_same_topk
from qvh_ctypes import Qvh

pytestmark = pytest.mark.gpu


def _check(oracle, base, q, k, metric, allowed=None):
    print(f"case: {base.shape} x {q.shape[0]} k={k} {metric} filtered={allowed is not None}", flush=True)
    stored = oracle.normalize(base) if metric == "cosine" else base
    idx = quiver.FlatIndex(base.shape[1], metric)
    idx.add(base)
    got_l, got_d = idx.search(q, k, filter=allowed)
    bm = None if allowed is None else rows_bitmap(allowed.astype(np.int64), base.shape[0])
    rows, dist = oracle.flat_search(stored, q, k, metric, bm)
    exp_l = rows.astype(np.int64)
    exp_l[rows == np.uint32(0xFFFFFFFF)] = -1
    assert_same_topk(got_l, got_d, exp_l, dist,
                     lambda qi, labels: oracle.flat_pair_dist(stored, q, np.full(labels.size, qi), labels, metric))


def _normal(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("dim", [1, 8, 16, 17, 24, 40, 64, 100, 120, 127, 128])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_row_widths(oracle, dim, metric):
    rng = np.random.default_rng(dim)
    _check(oracle, _normal(rng, 4_099, dim), _normal(rng, 45, dim), 10, metric)


@pytest.mark.parametrize("nq", [33, 128, 129, 256, 257, 512, 513, 1_025])
@pytest.mark.parametrize("k", [10, 21, 43])
def test_query_blocks_and_lists(oracle, nq, k):
    rng = np.random.default_rng(nq + k)
    base, q = _normal(rng, 9_000, 40), _normal(rng, nq, 40)
    _check(oracle, base, q, k, "l2")
    _check(oracle, np.round(40.0 * base), np.round(40.0 * q), k, "l2")


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 1_000, 1_041])
def test_row_counts_and_filters(oracle, n):
    rng = np.random.default_rng(n)
    base, q = _normal(rng, n, 20), _normal(rng, 300, 20)
    for k in (1, 11, 22):
        _check(oracle, base, q, k, "cosine")
        _check(oracle, base, q, k, "l2", np.arange(0, n, 3, dtype=np.uint64))


@pytest.mark.parametrize("rows_exp,query_exp", [(0, 0), (-40, 0), (40, 0), (0, -30), (0, 30), (-25, 25), (25, -25)])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_magnitudes(oracle, rows_exp, query_exp, metric):
    """Powers of two on either side, a spread of 2^12 between the queries of one batch, and a spread
    of 2^20 between the elements of a row."""
    rng = np.random.default_rng(7)
    base = np.ldexp(_normal(rng, 6_000, 33), rows_exp).astype(np.float32)
    base[:, :3] = np.ldexp(base[:, :3], -20)
    q = np.ldexp(_normal(rng, 140, 33), query_exp + rng.integers(-6, 7, (140, 1))).astype(np.float32)
    q[0] = 0.0
    _check(oracle, base, q, 10, metric)


@pytest.mark.parametrize("rows_exp,query_exp", [(-80, 60), (60, -80), (-80, -70), (-76, -76), (-74, -74), (-74, -148),
                                                (-84, -70), (-148, -148), (-140, 40)])
@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("dim", [16, 32, 136])
def test_magnitudes_whose_squares_underflow(oracle, rows_exp, query_exp, metric, dim):
    """Norms whose squares are subnormal or zero in float, beside normal ones on the other side: the
    16-bit scans (k = 10, 30), the fp32 scan (k = 50) and, for 8 queries, the ring scan."""
    rng = np.random.default_rng(11)
    base = np.ldexp(_normal(rng, 1_500, dim), rows_exp).astype(np.float32)
    q = np.ldexp(_normal(rng, 40, dim), query_exp).astype(np.float32)
    for k in (10, 30, 50):
        _check(oracle, base, q, k, metric)
    _check(oracle, base, q[:8], 10, metric)


@pytest.mark.parametrize("dim,k", [(16, 10), (40, 30), (136, 10)])
@pytest.mark.parametrize("rows_exp", [-50, -24, 0, 40])
def test_zero_queries_are_certified(oracle, dim, k, rows_exp):
    """A zero query's L2 distances are the rows' squared norms: no query may need the exact kernel."""
    rng = np.random.default_rng(dim)
    base = np.ldexp(_normal(rng, 1_500, dim), rows_exp).astype(np.float32)
    base *= rng.uniform(1.0, 2.0, (1_500, 1)).astype(np.float32)  # squared norms further apart than the bound
    q = np.zeros((40, dim), np.float32)
    idx = quiver.FlatIndex(dim, "l2")
    idx.add(base)
    print(f"case: {dim} {k} {rows_exp}", flush=True)
    labels, dist = idx.search(q, k)
    assert Qvh().last_fallbacks(idx._index._device_handle) == 0
    rows, exp = oracle.flat_search(base, q, k, "l2")
    assert np.array_equal(labels, rows.astype(np.int64)) and np.array_equal(dist.view(np.uint32), exp.view(np.uint32))


@pytest.mark.parametrize("top", [255, 2_048, 2_049, 4_000])
def test_integer_magnitudes(oracle, top):
    """Integers up to and above 2,048, up to which an fp16 value holds every integer."""
    rng = np.random.default_rng(top)
    base = rng.integers(-3, 4, (5_000, 24)).astype(np.float32)
    base[::7, 5] = top - rng.integers(0, 4, base[::7, 5].shape)
    q = rng.integers(-3, 4, (70, 24)).astype(np.float32)
    q[:40, 5] = top - rng.integers(0, 4, 40)
    _check(oracle, base, q, 10, "l2")


@pytest.mark.parametrize("row", [0, 32_767, 32_768, 70_000])
@pytest.mark.parametrize("value", [0.3, 3_000.0])
def test_one_row_decides_the_bound(oracle, row, value):
    """One row that is no small integer, or above 2,048, among many that are: the store's bound data must
    see it wherever the work-groups that collect them come to it (32,768 rows a step)."""
    rng = np.random.default_rng(row)
    base = rng.integers(-9, 10, (70_001, 16)).astype(np.float32)
    base[row, 3] = value
    q = rng.integers(-9, 10, (40, 16)).astype(np.float32)
    q[:8, 3] = value
    _check(oracle, base, q, 10, "l2")


def test_equal_rows(oracle):
    """Every row stored 40 times: equal distances in row order, inside a group and across groups."""
    rng = np.random.default_rng(3)
    base = np.round(20.0 * _normal(rng, 300, 16))
    q = np.round(20.0 * _normal(rng, 200, 16))
    _check(oracle, np.repeat(base, 40, axis=0), q, 10, "l2")
    _check(oracle, np.tile(base, (40, 1)), q, 10, "l2")


@pytest.mark.parametrize("dim", [129, 144, 145, 160, 161, 300, 1_000])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_wide_row_widths(oracle, dim, metric):
    rng = np.random.default_rng(dim)
    base, q = _normal(rng, 3_001, dim), _normal(rng, 77, dim)
    _check(oracle, base, q, 10, metric)
    _check(oracle, base, q, 40, metric)


@pytest.mark.parametrize("nq", [33, 63, 64, 65, 255, 256, 257, 600])
@pytest.mark.parametrize("n", [1, 16, 255, 256, 257, 2_000])
def test_wide_blocks_and_filters(oracle, nq, n):
    rng = np.random.default_rng(nq * n)
    base, q = _normal(rng, n, 130), np.ldexp(_normal(rng, nq, 130), rng.integers(-6, 7, (nq, 1))).astype(np.float32)
    _check(oracle, base, q, 11, "l2")
    _check(oracle, base, q, 25, "cosine")
    _check(oracle, base, q, 10, "l2", np.arange(0, n, 3, dtype=np.uint64))
    _check(oracle, np.round(2.0 * base), np.round(2.0 * q / np.abs(q).max()), 10, "l2")


@pytest.mark.parametrize("nq,n,dim,k", [(600, 2_000, 768, 43), (768, 2_000, 768, 43), (769, 2_000, 768, 43),
                                        (1_025, 3_000, 1_040, 43), (1_025, 700, 1_040, 21), (1_025, 12_000, 520, 25),
                                        (1_025, 2_000, 768, 11)])
def test_wide_large_batches(oracle, nq, n, dim, k):
    """Batches past the merge's four waves a query, on both sides of the rule that gives few wide rows to
    the fp32 scan; with listed rows too."""
    rng = np.random.default_rng(n + k)
    base, q = _normal(rng, n, dim), _normal(rng, nq, dim)
    _check(oracle, base, q, k, "l2")
    if k <= 21:
        _check(oracle, base, q, k, "ip", np.arange(0, n, 2, dtype=np.uint64))
