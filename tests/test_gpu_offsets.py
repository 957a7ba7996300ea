"""The value offsets' chunks of 2048 values (k_sort_begin, launch_offsets): fields of every remainder in
one batch, each with the extremes that its offset is made of in its first and last value, and one large
field among thousands of small ones."""
import numpy as np
import pytest

from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


def _field(size, n):
    return dict(sigma=2.0, x0=np.zeros(2), step=1.0, size=size, n=n, num_iter=4, max_dist=3.5)


def _same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


@pytest.mark.parametrize('precision', ['fp32c', 'fp64'])
@pytest.mark.parametrize('counts', [[1, 2047, 2048, 2049, 1, 1, 9000, 4096, 3], [8193], [2048 * 5, 2048 * 4, 1],
                                    [1, 1, 1, 10240, 1], [12287, 12288, 12289, 2047]])
def test_chunks(precision, counts):
    rng = np.random.default_rng(sum(counts))
    size = (40, 40)
    pts = [rng.uniform(0.0, 39.0, (n, 2)) for n in counts]
    val = [rng.normal(0.0, 1.0, n) for n in counts]
    for i, v in enumerate(val):
        v[0], v[-1] = -1e6 * (i + 1), 3e6 * (i + 1)
    got = BarnesBatch([_field(size, n) for n in counts], precision=precision).interpolate(pts, val)
    for n, p, v, g in zip(counts, pts, val, got):
        assert _same(g, BarnesBatch([_field(size, n)], precision=precision).interpolate([p], [v])[0])


def test_large_field_among_small_ones():
    """4100 chunks and 4200 fields: a chunk grid of fields times the largest field's chunks would have
    2^24 workgroups of 256."""
    rng = np.random.default_rng(11)
    n, small = 4100 * 2048, [3] * 4200
    pts = [rng.uniform(0.0, 11.0, (k, 2)) for k in small]
    val = [rng.normal(10.0, 1.0, k) for k in small]
    alone = BarnesBatch([_field((12, 12), k) for k in small], precision='fp32c').interpolate(pts, val)
    big = rng.uniform(0.0, 2047.0, (n, 2)), rng.normal(10.0, 1.0, n)
    batch = BarnesBatch([_field((12, 12), k) for k in small] + [_field((2048, 2048), n)], precision='fp32c')
    got = batch.interpolate(pts + [big[0]], val + [big[1]])
    assert all(_same(a, b) for a, b in zip(alone, got))
    # 2 points to a cell and a wide kernel: the field is flat at the values' mean (sigma 1 / sqrt(n))
    assert abs(np.nanmean(got[-1]) - 10.0) < 1e-2
