"""The sort stage (k_field_sort; k_sort_begin, k_point_keys, k_scan_tiles, k_row_scatter, k_row_sort) at
its edges: point counts around the threads' shares, rows around 4096, rows' entries around every limit of
the row sorts, more than one scan tile, one workgroup's rows in several rounds.

The list's order decides the order of the injection's sums, so the order is checked through results
that must be equal bit for bit: the FP64 injection against the oracle's point loop, and FP32C fields
alone (one workgroup sorts) against the same fields in a batch with one that forces row buckets."""
import numpy as np
import pytest

from fastbarnes import interpolation
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu

FN = {1: interpolation._inject_data_1d, 2: interpolation._inject_data_2d, 3: interpolation._inject_data_3d}


def _points(rng, size, counts):
    """counts[k] points with base row k (x-lines in order), shuffled; columns crowded enough to meet."""
    dim = len(size)
    row = np.repeat(np.arange(len(counts)), counts)
    n = len(row)
    c = rng.uniform(0.0, 0.999, (n, dim))
    c[:, 0] += rng.integers(0, max(1, min(size[0] - 1, 23)), n)
    if dim >= 2:
        c[:, 1] += row % (size[1] - 1)
    if dim >= 3:
        c[:, 2] += row // (size[1] - 1)
    rng.shuffle(c)
    return c


CASES = [((40, 50), [k] * 3 + [0, 1]) for k in (1, 2, 3, 4, 5, 8, 9, 16, 17, 63, 64, 65, 128, 256, 257, 1024, 1025)] + [
    ((40, 50), [8191]), ((40, 50), [8192]), ((40, 50), [8193]), ((40, 50), [9000, 1, 2]),
    ((33, 40), [1023]), ((33, 40), [31] * 33), ((33, 40), [105] * 38 + [4]),
    ((7, 4096), [2] * 4095), ((7, 4097), [2] * 4096), ((5, 9000), [1, 0, 20] * 2900),
    ((6, 65, 63), [1] * 300 + [70]), ((6, 65, 64), [3, 0, 18] * 900), ((9, 700, 800), [2, 0, 17, 0] * 900),
    ((9000,), [5000]), ((9000,), [20000]),
]


@pytest.mark.parametrize('size,counts', CASES)
def test_list_order_bitwise(orc, size, counts):
    dim = len(size)
    rng = np.random.default_rng(sum(counts) + sum(size))
    pts = _points(rng, size, counts)
    n = len(pts)
    pts = np.concatenate([pts, rng.uniform(-3.0, -1.0, (3, dim))])   # dropped points
    order = rng.permutation(n + 3)
    pts, val = pts[order], rng.normal(0.0, 1.0, n + 3) * np.exp(rng.uniform(-10, 10, n + 3))
    x0, step = np.zeros(dim), np.ones(dim)
    vg, wg = np.zeros(size[::-1]), np.zeros(size[::-1])
    rv, rw = vg.copy(), wg.copy()
    FN[dim](vg, wg, pts, val, x0, step, size)
    orc.inject_raw(rv, rw, pts, val, x0, step, size)
    assert np.array_equal(vg.view(np.uint64), rv.view(np.uint64))
    assert np.array_equal(wg.view(np.uint64), rw.view(np.uint64))


@pytest.mark.parametrize('precision', ['fp32c', 'fp64'])
@pytest.mark.parametrize('n', [1, 63, 1024, 1025, 2049, 5000, 8189, 8192])
def test_both_sorts_give_the_same_fields(precision, n):
    rng = np.random.default_rng(n + 1)
    sizes = [(64, 50), (61, 33), (48, 48)]
    fs = []
    for i, m in enumerate([n, 1 if n % 2 else 40, 300]):
        size = sizes[i]
        pts = rng.uniform(-0.5, np.asarray(size) - 0.5, (m, 2))
        pts[rng.random(m) < 0.3] = rng.uniform(3.0, 5.0, (1, 2))
        val = rng.normal(7.0, 3.0, m)
        if i == 2:
            val[17] = np.nan   # the field's offset, and with it every node, becomes NaN
        fs.append((pts, val, size))
    big = (rng.uniform(0.0, 30.0, (9000, 2)), rng.normal(0.0, 1.0, 9000), (32, 32))

    def run(group):
        batch = BarnesBatch([dict(sigma=2.0, x0=np.zeros(2), step=1.0, size=s, n=len(v), num_iter=4, max_dist=3.5)
                             for _, v, s in group], precision=precision)
        return batch.interpolate([p for p, _, _ in group], [v for _, v, _ in group])
    few, many = run(fs), run(fs + [big])
    for (_, v, _), a, b in zip(fs, few, many):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)) or (
            np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)]))
        assert bool(np.isnan(a).all()) == bool(np.isnan(v).any())
