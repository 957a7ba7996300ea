"""Naive sums whose nodes lie mostly far from every station (k_naive_finish): the oracle's sums in every
layout of the products, and no longer than node by node.

Tolerance: weights down to exp(-685) (37 sigma) are normal numbers; the rounding of their argument is 685 *
2^-53 of the weight (test_gpu_naive.py), 1e-12 of the values' range.  From 39.5 sigma on every weight is 0."""
import time

import numpy as np
import pytest

from fastbarnes import interpolation

pytestmark = pytest.mark.gpu


def _corner(n, spread, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(0.0, spread, (n, 2)), rng.normal(0.0, 1.0, n)


# parts: fewer than 512 tiles of 64 x 64 nodes; none: 512 tiles and one block of stations; several blocks
@pytest.mark.parametrize('size,n', [((600, 300), 300), ((130, 90), 700), ((2049, 1030), 40), ((9000, 70), 1200)])
def test_far_nodes(orc, size, n):
    sigma, step = 0.1, 9.0 / size[0]
    pts, val = _corner(n, 0.6, n)
    out = interpolation.barnes(pts, val, sigma, 0.0, step, size, method='naive')
    ref = orc.interpolate_naive(pts, val, np.full(2, sigma), np.zeros(2), np.full(2, step), size)
    x, y = step * np.arange(size[0]), step * np.arange(size[1])
    d2 = np.full(size[::-1], np.inf)
    for k in range(n):
        np.minimum(d2, (x[None, :] - pts[k, 0]) ** 2 + (y[:, None] - pts[k, 1]) ** 2, out=d2)
    d = np.sqrt(d2) / sigma
    near, far = d < 37.0, d > 39.5
    assert (near & (d > 36.5)).any() and far.any()
    assert not np.isnan(ref[near]).any() and np.abs(out - ref)[near].max() <= 1e-12 * np.ptp(val)
    assert np.isnan(out[far]).all() and np.isnan(ref[far]).all()


def _best(fn, reps):
    fn()
    best = np.inf
    for _ in range(reps):
        t = time.perf_counter()
        fn()
        best = min(best, time.perf_counter() - t)
    return best


def test_far_nodes_time():
    """As many nodes in 15 rows are summed node by node."""
    pts, val = _corner(3490, 4.0, 1)
    run = lambda size: interpolation.barnes(pts, val, 0.25, 0.0, 75.0 / size[0], size, method='naive')
    assert _best(lambda: run((600, 300)), 5) < 1.1 * _best(lambda: run((12000, 15)), 5)


def test_few_stations_time():
    """One station: one launch, as for as many nodes in 15 rows."""
    pts, val = np.array([[20.0, 10.0]]), np.array([3.0])
    run = lambda size: interpolation.barnes(pts, val, 5.0, 0.0, 1.0, size, method='naive')
    assert _best(lambda: run((64, 64)), 30) < 1.25 * _best(lambda: run((273, 15)), 30)


@pytest.mark.parametrize('size,n', [((17, 19), 172), ((17, 19), 173), ((65, 129), 179), ((600, 300), 105),
                                    ((600, 300), 106), ((33, 40, 35), 181)])
def test_both_sides_of_few(orc, size, n):
    """No weight below exp(-2 * 3): 50 ulp of a weight's rounding and its products, as in
    test_gpu_naive.py, are 1e-14 of the values' range."""
    rng = np.random.default_rng(n)
    pts, val = rng.uniform(0.0, 1.0, (n, len(size))) * np.asarray(size), rng.normal(3.0, 2.0, n)
    out = interpolation.barnes(pts, val, 300.0, 0.0, 1.0, size, method='naive')
    ref = orc.interpolate_naive(pts, val, np.full(len(size), 300.0), np.zeros(len(size)), np.ones(len(size)), size)
    assert np.abs(out - ref).max() <= 1e-14 * np.ptp(val)
