"""Single calls on host arrays (the pinned staging of fb_api.hip) give the bits of a plan on device
buffers where the points leave the descriptors little room in the block's first megabyte, or none."""
import numpy as np
import pytest

from fastbarnes import interpolation
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def _field(size, n, seed):
    rng = np.random.default_rng(seed)
    pts = rng.uniform(-0.1, 1.1, (n, len(size))) * np.asarray(size) * 0.125
    return pts, rng.normal(10.0, 2.0, n), dict(sigma=1.0, x0=0.0, step=0.125, size=size, num_iter=4, max_dist=3.5)


# n points of dimension d take 8 n (d + 1) bytes, rounded up per array, of 1048576: room for every
# descriptor, for the first ones only, for none, and for the points or their values alone
@pytest.mark.parametrize('precision', ['fp64', 'fp32c'])
@pytest.mark.parametrize('size,n', [((2400, 1200), 41000), ((2400, 1200), 43000), ((1200, 600), 43600),
                                    ((1200, 600), 43680), ((600, 300), 43700), ((600, 300), 70000),
                                    ((100, 90, 60), 32000), ((100, 90, 60), 32700), ((100, 90, 60), 32768)])
def test_points_fill_the_block(precision, size, n):
    pts, val, c = _field(size, n, n)
    got = interpolation.barnes(pts, val, precision=precision, **c)
    ref = BarnesBatch([dict(c, n=n)], precision=precision).interpolate([pts], [val])[0]
    assert _same(got, ref)
