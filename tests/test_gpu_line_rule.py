"""FP64 line passes on both sides of the rules between LDS rings, of more or fewer iterations to a launch, and a
thread per line (AxisLines): the oracle's bits, and short columns of a large grid in a time that fits their bytes."""
import numpy as np
import pytest

from fastbarnes.batched import BarnesBatch
from fastbarnes import hip

pytestmark = pytest.mark.gpu


def _field(size, n, num_iter, halves):
    """A field whose half kernels are halves[a]: sigma^2 of that width plus 0.4, in steps of 1."""
    sigma = [np.sqrt(((2 * (t + 0.4) + 1) ** 2 - 1) * num_iter / 12.0) for t in halves]
    return dict(sigma=sigma, x0=[0.0] * len(size), step=1.0, size=size, n=n, num_iter=num_iter, max_dist=3.5)


def _check(orc, fields, seed):
    rng = np.random.default_rng(seed)
    pts = [rng.uniform(-0.02, 1.02, (f['n'], len(f['size']))) * np.asarray(f['size']) for f in fields]
    val = [rng.normal(10.0, 2.0, f['n']) for f in fields]
    out = BarnesBatch(fields, precision='fp64').interpolate(pts, val)
    for f, p, v, o in zip(fields, pts, val, out):
        d = len(f['size'])
        ref = orc.interpolate_convol(p, v, np.asarray(f['sigma']), np.zeros(d), np.ones(d), f['size'],
                                     num_iter=f['num_iter'], max_dist=f['max_dist'])
        assert np.array_equal(np.isnan(o), np.isnan(ref))
        ok = ~np.isnan(ref)
        assert ok.any() and np.array_equal(o[ok].view(np.uint32), ref[ok].view(np.uint32))


# columns of 6 to 24 nodes in grids large and small; odd counts of iterations end in the other buffer
@pytest.mark.parametrize('size,num_iter,halves', [
    ((1001, 503, 6), 4, (1, 1, 1)), ((601, 6, 301), 5, (1, 1, 1)), ((300, 299, 16), 1, (2, 2, 2)),
    ((5, 301, 299), 4, (1, 1, 1)), ((6, 501, 333), 9, (0, 1, 1)), ((16, 101, 307), 8, (3, 1, 1)),
    ((17, 101, 307), 8, (3, 1, 1)), ((40, 70001), 8, (2, 1)), ((64, 401, 250), 6, (2, 2, 30)),
    ((100001, 12), 3, (1, 2)), ((70000, 24), 8, (2, 7)), ((40, 31, 6), 4, (1, 1, 1))])
def test_short_columns_bitwise(orc, size, num_iter, halves):
    _check(orc, [_field(size, 400, num_iter, halves)], size[0])


def test_many_small_fields_bitwise(orc):
    sizes = [(30, 20), (25, 17), (33, 8)]
    _check(orc, [_field(sizes[k % 3], 30, 3 + k % 4, (2, 1 + k % 2)) for k in range(900)], 5)


@pytest.mark.parametrize('halves', [(3, 2), (170, 300)])
def test_mixed_iterations_bitwise(orc, halves):
    """More iterations than a launch takes (8; with a half kernel of 300 two) and fewer in one plan: the
    fields' quotients are formed by different launches of the last axis."""
    size = (700, 690) if halves[0] > 100 else (61, 47)
    _check(orc, [_field(size, 200, k, halves) for k in (3, 8, 9, 1, 12)], 11)


def _times(f):
    rng = np.random.default_rng(1)
    pts = hip.DeviceArray.from_numpy(rng.uniform(0.0, 1.0, (f['n'], len(f['size']))) * np.asarray(f['size']))
    val = hip.DeviceArray.from_numpy(rng.normal(0.0, 1.0, f['n']))
    batch = BarnesBatch([f], precision='fp64')
    out = hip.DeviceArray((batch.total_out,), np.float32)
    s = hip.Stream()
    batch.set_timing(True)
    best = {}
    for _ in range(5):
        batch.execute(pts.ptr, val.ptr, out.ptr, s.ptr)
        s.synchronize()
        for k, ms in batch.stage_times().items():
            best[k] = min(best.get(k, ms), ms)
    return best


def test_short_columns_time():
    """z lines of 6 nodes: through rings they took 34 times the x lines of the same cells."""
    best = _times(_field((1000, 1000, 6), 2000, 4, (1, 1, 1)))
    assert best['lines_z'] + best['finalize'] < 12.0 * best['lines_x']


def test_short_rows_time():
    """x lines of 30 nodes at 8 iterations: all in one launch they took 5.4 times as long as at 4."""
    x = [_times(_field((30, 128000), 2000, it, (1, 1)))['lines_x'] for it in (4, 8)]
    assert x[1] < 3.5 * x[0]
