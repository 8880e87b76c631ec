"""The error bound that the 16-bit flat scans' certificate rests on, measured: single matrix steps
(v_mfma_f32_32x32x16_f16) against 64-bit sums, at most 18 u of the sum of their magnitudes (u = 2^-24), in
which a half below the normal range counts as the smallest normal one, and exact on integers below
2^24, and the group minima that the scans list against 64-bit distances, at
most the bound of scan_bound (flat_half.hpp), which also covers the reference's own rounding."""

import ctypes as C
import os

import numpy as np
import pytest

from qvh_ctypes import ROOT

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
_vp = C.c_void_p


@pytest.fixture(scope="module")
def probe():
    L = C.CDLL(os.path.join(ROOT, "tests", "cpp", "libhalf_scan_probe.so"))
    L.probe_matrix_steps.argtypes = [_vp, _vp, _vp, _vp, C.c_uint32]
    L.probe_half_minima.argtypes = [_vp, _vp, C.c_uint64, C.c_uint32, _vp, _vp, _vp, C.c_uint32, C.c_int, _vp, C.c_int,
                                    C.c_int, C.c_int, C.c_uint64, _vp, _vp, _vp]
    return L


def _p(a):
    return a.ctypes.data_as(_vp)


def _steps(L, a, b, c):
    a, b, c = a.astype(np.float16), b.astype(np.float16), np.ascontiguousarray(c, np.float32)
    d = np.empty_like(c)
    assert L.probe_matrix_steps(_p(a), _p(b), _p(c), _p(d), a.shape[0]) == 0
    a, b = a.astype(np.float64), b.astype(np.float64)
    exact = a @ b.transpose(0, 2, 1) + c
    # The unit aligns a product by its operands' exponents, and a subnormal half has the exponent of the
    # smallest normal one, 2^-14.
    a, b = np.maximum(np.abs(a), 2.0 ** -14), np.maximum(np.abs(b), 2.0 ** -14)
    return d.astype(np.float64), exact, a @ b.transpose(0, 2, 1) + np.abs(c)


@pytest.mark.parametrize("spread", [0, 4, 10, 14])
@pytest.mark.parametrize("kind", ["plain", "cancelling", "subnormal", "large sum before"])
def test_matrix_step_error(probe, kind, spread):
    rng = np.random.default_rng(spread)
    shape = (256, 32, 16)
    a = np.ldexp(rng.uniform(1, 2, shape) * rng.choice([-1, 1], shape), rng.integers(-spread, 1, shape))
    b = np.ldexp(rng.uniform(1, 2, shape) * rng.choice([-1, 1], shape), rng.integers(-spread, 1, shape))
    c = np.ldexp(rng.standard_normal((256, 32, 32)), rng.integers(-2 * spread, 3, (256, 32, 32)))
    if kind == "cancelling":  # every second product takes the one before it back, up to a bit
        a[:, :, 1::2], b[:, :, 1::2] = -a[:, :, ::2], b[:, :, ::2] * (1 + 2.0 ** -10)
    elif kind == "subnormal":
        a = np.ldexp(a, -16)
        c = np.ldexp(c, -16)
    elif kind == "large sum before":
        c = np.ldexp(c, 12)
    print(f"case: matrix steps {kind} spread={spread}", flush=True)
    got, exact, size = _steps(probe, a, b, c)
    worst = float((np.abs(got - exact) / (U * size)).max())
    print(f"worst error {worst:.2f} u of the sum of magnitudes")
    assert worst <= 18.0


@pytest.mark.parametrize("top", [1, 40, 700, 1_000])
def test_matrix_step_is_exact_on_integers(probe, top):
    """16 products and the sum before them below 2^24 in all."""
    rng = np.random.default_rng(top)
    a, b = rng.integers(-top, top + 1, (256, 32, 16)), rng.integers(-top, top + 1, (256, 32, 16))
    c = rng.integers(-(2 ** 24 - 1 - 16 * top * top), 2 ** 24 - 16 * top * top, (256, 32, 32))
    print(f"case: integer matrix steps top={top}", flush=True)
    got, exact, _ = _steps(probe, a, b, c)
    assert np.array_equal(got, exact)


FORMS = [  # kl, products, two lanes a query, rows a split
    (16, 3, 0, 256), (16, 3, 1, 256), (32, 3, 1, 512)]


def _minima(L, x, q, l2, kl, products, pair, rows):
    """(minima, 64-bit minima, bounds): the first two [nq, groups]."""
    n, dp = x.shape
    nq = q.shape[0]
    wide = dp > 128
    x64, q64 = x.astype(np.float64), q.astype(np.float64)
    xn, qn = (x64 * x64).sum(1).astype(np.float32), (q64 * q64).sum(1).astype(np.float32)
    meta = np.array([xn.max(), 0, np.abs(x).max(), 0], np.float32).view(np.uint32)
    lists = n // rows * (2 if wide or pair else 1)
    d, g = np.empty((nq, lists, kl), np.float32), np.empty((nq, lists, kl), np.uint32)
    bound = np.empty(nq)
    qlen = np.sqrt((q64 * q64).sum(1))
    st = L.probe_half_minima(_p(x), _p(xn), n, dp, _p(q), _p(qn), _p(qlen), nq, int(l2), _p(meta), kl, products, pair, rows,
                             _p(d), _p(g), _p(bound))
    assert st == 0
    got = np.full((nq, n // 16), np.nan)
    held = g.reshape(nq, -1) != np.uint32(0xFFFFFFFF)
    assert (held.sum(1) == n // 16).all()
    for i in range(nq):
        got[i, g[i].reshape(-1)[held[i]]] = d[i].reshape(-1)[held[i]]
    if l2:
        true = np.stack([((x64 - v) ** 2).sum(1) for v in q64])
    else:
        true = 1.0 - q64 @ x64.T
    return got, true.reshape(nq, -1, 16).min(2), bound


@pytest.mark.parametrize("dp", [16, 24, 64, 104, 128, 144, 304, 1_024])
@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("rows_exp,query_exp", [(0, 0), (-40, 0), (40, 0), (0, 30), (-25, 25), (-50, -52), (-80, 55)])
def test_scan_minima_within_the_bound(probe, dp, metric, rows_exp, query_exp):
    rng = np.random.default_rng(dp)
    worst = 0.0  # every squared norm is within float's range: past it the search has no bound
    for kl, products, pair, rows in FORMS:
        if dp > 128:
            rows = 512 if kl == 16 else 1_024
            if kl == 16 and pair:
                continue
        x = np.ldexp(rng.standard_normal((4 * rows, dp)), rows_exp).astype(np.float32)
        x[::3, : dp // 2] = np.ldexp(x[::3, : dp // 2], -18)  # far smaller elements in some rows
        q = np.ldexp(rng.standard_normal((70, dp)), query_exp).astype(np.float32)
        q[:20] = np.ldexp(x[:20], query_exp - rows_exp)  # near rows: the difference cancels
        q[20] = 0.0
        print(f"case: minima {dp} {metric} {rows_exp} {query_exp} lists of {kl} pair={pair}", flush=True)
        got, true, bound = _minima(probe, x, q, metric == "l2", kl, products, pair, rows)
        error = np.abs(got - true) / bound[:, None]
        worst = max(worst, float(error.max()))
    print(f"worst error {worst:.4f} of the bound")
    assert worst <= 1.0


@pytest.mark.parametrize("dp", [16, 64, 128])
@pytest.mark.parametrize("top", [5, 100, 255, 2_048])
def test_scan_minima_are_exact_on_integers(probe, dp, top):
    """One product of halves, (P + R)^2 below 2^24."""
    rng = np.random.default_rng(top)
    x, q = (rng.integers(-5, 6, (s, dp)).astype(np.float32) for s in (512, 70))
    x[:, 0], q[:, 0] = rng.integers(-top // 2, top // 2 + 1, 512), rng.integers(-top // 2, top // 2 + 1, 70)
    x[::9, 0], q[::9, 0] = top if top < 2_048 else 2_000, top // 2 if top < 2_048 else 2_000
    print(f"case: integer minima {dp} {top}", flush=True)
    got, true, _ = _minima(probe, x, q, True, 10, 1, 0, 128)
    assert np.array_equal(got, true)
