"""k-means with its means on the device, at the sizes where the update kernel's split changes: widths
around its 64- and 128-dim blocks, point counts around the 1,024 assignments of a scan step, clusters
larger than its 2,048-point list, empty clusters (split on the host), the host's own sums past 256
centroids a dimension, and sub-spaces trained together. Centroids must equal the oracle's bit for
bit (the sums run in double in point order on both sides)."""

import numpy as np
import pytest

import quiver_amd as quiver

pytestmark = pytest.mark.gpu


def _same(oracle, x, k, iterations, **kw):
    print(f"case: {x.shape} k={k} iterations={iterations} {kw}", flush=True)
    got = quiver.kmeans(x, k, iterations, **kw)
    exp = oracle.kmeans(x, k, iterations, **kw)
    assert np.array_equal(got.view(np.uint32), exp.reshape(got.shape).view(np.uint32))


@pytest.mark.parametrize("dim", [1, 4, 63, 64, 65, 127, 128, 129, 300])
def test_widths(oracle, dim):
    x = np.random.default_rng(dim).standard_normal((3_000, dim)).astype(np.float32)
    _same(oracle, x, 20, 4, seed=dim)


@pytest.mark.parametrize("n", [1, 5, 63, 64, 1_023, 1_024, 1_025, 2_049])
def test_point_counts(oracle, n):
    x = np.random.default_rng(n).standard_normal((n, 6)).astype(np.float32)
    _same(oracle, x, min(n, 5), 3)


@pytest.mark.parametrize("k", [1, 2, 300, 600])
def test_large_clusters_and_many_centroids(oracle, k):
    """k = 1 and 2: one list holds thousands of points; k = 300 and 600 over 1 and 2 dims: the host's sums."""
    rng = np.random.default_rng(k)
    x = rng.standard_normal((9_000, 1 if k == 300 else 2)).astype(np.float32)
    _same(oracle, x, k, 4, max_points_per_centroid=10_000)


def test_empty_clusters_and_iterations(oracle):
    x = np.zeros((2_000, 3), np.float32)
    x[:30] = np.random.default_rng(1).standard_normal((30, 3))
    for iterations in (0, 1, 2, 7):
        _same(oracle, x, 64, iterations)


@pytest.mark.parametrize("dim,m", [(8, 8), (24, 6), (132, 2)])
def test_sub_spaces_together(oracle, dim, m):
    """All sub-spaces of a product quantizer in one set of launches; constant columns leave most of a
    sub-space's clusters empty."""
    x = np.random.default_rng(dim).standard_normal((1_500, dim)).astype(np.float32)
    x[:, : dim // m] = 0.0
    x[:200, 0] = np.arange(200)
    idx = quiver.IvfPqIndex(dim, "l2", nlist=8, m=m, train_iterations=5)
    print(f"case: train {dim} {m}", flush=True)
    idx.train(x)
    cent, cb, _ = oracle.ivfpq_train(x, "l2", 8, m, 5, 1234)
    assert np.array_equal(idx.centroids.view(np.uint32), cent.view(np.uint32))
    assert np.array_equal(idx.codebook.view(np.uint32), cb.view(np.uint32))


@pytest.mark.parametrize("dim,k", [(2, 64), (4, 256), (8, 64), (16, 40), (40, 8), (64, 8), (128, 3)])
@pytest.mark.parametrize("share", [0.0, 0.5, 0.97])
def test_dominating_clusters(oracle, dim, k, share):
    """One cluster that holds a share of the points: the means are taken on the device, on the host, or on
    the host from the first iteration that meets too large a cluster."""
    rng = np.random.default_rng(dim + k)
    x = rng.standard_normal((6_000, dim)).astype(np.float32)
    x[: int(share * 6_000)] = 50.0 + 0.01 * x[: int(share * 6_000)]
    x = x[rng.permutation(6_000)]
    _same(oracle, x, k, 6, max_points_per_centroid=10_000)


@pytest.mark.parametrize("m", [2, 8, 16])
def test_dominating_clusters_in_sub_spaces(oracle, m):
    x = np.random.default_rng(m).standard_normal((1_500, 4 * m)).astype(np.float32)
    x[:1_200, :4] = 7.0
    x[:700, 4:8] = -3.0
    idx = quiver.IvfPqIndex(4 * m, "l2", nlist=4, m=m, train_iterations=5)
    print(f"case: train {m}", flush=True)
    idx.train(x)
    cent, cb, _ = oracle.ivfpq_train(x, "l2", 4, m, 5, 1234)
    assert np.array_equal(idx.centroids.view(np.uint32), cent.view(np.uint32))
    assert np.array_equal(idx.codebook.view(np.uint32), cb.view(np.uint32))
