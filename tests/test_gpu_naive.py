"""The naive sums as matrix products (fb_naive.hip) against the oracle's node-by-node sums, at the
edges of their tiles (64 nodes), station groups (4) and splits, and where the weights underflow.

Tolerance: a weight exp(-d) carries the rounding of d (d <= 40 for every weight that counts beside
the largest of its node within 1e-17) and of two products, so each sum is within about 50 ulp
of the other's, 1e-14 relative, and the quotient within 2e-14 of the values' range."""
import numpy as np
import pytest

from fastbarnes import interpolation

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16), (17, 15), (63, 65), (64, 64), (65, 129), (200, 31), (16, 4, 4), (33, 9, 7), (64, 16, 5)]


@pytest.mark.parametrize('size', SHAPES)
@pytest.mark.parametrize('n', [1, 3, 64, 257, 1501])
def test_naive_products(orc, size, n):
    dim = len(size)
    rng = np.random.default_rng(n + sum(size))
    step, x0 = 0.25, np.full(dim, -3.0)
    pts = x0 + rng.uniform(-0.1, 1.1, (n, dim)) * np.asarray(size) * step
    val = rng.normal(3.0, 2.0, n)
    sigma = np.array([0.9, 1.3, 0.7])[:dim]
    out = interpolation.barnes(pts, val, sigma, x0, step, size, method='naive')
    ref = orc.interpolate_naive(pts, val, sigma, x0, np.full(dim, step), size)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.max(np.abs(out - ref)[ok], initial=0.0) <= 2e-14 * max(1.0, np.ptp(val)) + 4 * np.spacing(np.abs(ref[ok]).max())


def test_naive_underflow(orc):
    """Stations in one corner of a field 90 sigma wide: products of factors that underflow one by
    one, sums below the smallest double (NaN), and ordinary nodes."""
    rng = np.random.default_rng(5)
    pts = rng.uniform(0.0, 0.4, (40, 2))
    val = rng.normal(0.0, 1.0, 40)
    size = (120, 110)
    out = interpolation.barnes(pts, val, 0.1, 0.0, 0.08, size, method='naive')
    ref = orc.interpolate_naive(pts, val, np.full(2, 0.1), np.zeros(2), np.full(2, 0.08), size)
    assert 0 < np.isnan(ref).sum() < ref.size
    far = orc.interpolate_naive(pts, np.ones(40), np.full(2, 0.1), np.zeros(2), np.full(2, 0.08), size)
    assert far.shape == ref.shape
    # the smallest weights are denormal, where one unit is the whole weight: compare where the
    # nearest station is within 37 sigma (weights over exp(-685))
    x, y = np.meshgrid(0.08 * np.arange(size[0]), 0.08 * np.arange(size[1]))
    d = np.sqrt(((x[..., None] - pts[:, 0]) ** 2 + (y[..., None] - pts[:, 1]) ** 2).min(-1)) / 0.1
    near = d < 37.0
    assert not np.isnan(ref[near]).any() and not np.isnan(out[near]).any()
    # at 37 sigma the argument's rounding is 685 * 2^-53 relative to the weight
    assert np.abs(out - ref)[near].max() <= 1e-12 * np.ptp(val)
    assert np.isnan(out[d > 39.5]).all() and np.isnan(ref[d > 39.5]).all()
