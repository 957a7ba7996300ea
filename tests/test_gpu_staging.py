"""Single calls on host arrays (the pinned staging of fb_api.hip) give the bits of a plan on device
buffers where the points leave the descriptors little room in the block's first megabyte, or none."""
import threading

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


def test_refused_calls_beside_good_ones():
    """A call that is refused after its first upload (no FP32C line pass takes half kernels of 3000)
    gives its blocks back while another thread's calls take blocks of the same sizes."""
    pts, val, c = _field((300, 150), 3000, 1)
    ref = BarnesBatch([dict(c, n=3000)], precision='fp32c').interpolate([pts], [val])[0]
    bad = dict(c, sigma=6928.0, step=2.0, size=(16000, 40))
    refused, good = [], []

    def refuse():
        for _ in range(50):
            try:
                interpolation.barnes(pts, val, precision='fp32c', **dict(bad, sigma=(6928.0, 4.0)))
            except RuntimeError as e:
                refused.append(str(e))

    t = threading.Thread(target=refuse)
    t.start()
    for _ in range(50):
        good.append(_same(interpolation.barnes(pts, val, precision='fp32c', **c), ref))
    t.join()
    assert len(refused) == 50 and all('fit no FP32C line pass' in e for e in refused)
    assert all(good)


@pytest.mark.parametrize('size,method', [((2600, 1700), 'optimized_convolution'), ((4099, 2053), 'convolution'),
                                         ((2048, 2048), 'optimized_convolution')])
def test_results_of_several_rounds(size, method):
    """Results of more than the 16 MB of the block's slots come down in rounds (16 MB exactly: in one)."""
    pts, val, c = _field(size, 3000, size[0])
    got = interpolation.barnes(pts, val, method=method, **c)
    ref = BarnesBatch([dict(c, n=3000, method=method)], precision='fp64').interpolate([pts], [val])[0]
    assert _same(got, ref)


def test_concurrent_callers():
    """More callers at once than idle blocks are kept, with results of one slot and of several."""
    sizes = [(300, 150), (1200, 600), (2400, 1200), (600, 300)]
    cases = []
    for k, size in enumerate(sizes):
        pts, val, c = _field(size, 2000 + 500 * k, k)
        ref = BarnesBatch([dict(c, n=len(val))], precision='fp64').interpolate([pts], [val])[0]
        cases.append((pts, val, c, ref))
    good = [0] * len(cases)

    def call(k):
        pts, val, c, ref = cases[k]
        for _ in range(12):
            good[k] += _same(interpolation.barnes(pts, val, **c), ref)

    threads = [threading.Thread(target=call, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert good == [12] * len(cases)
