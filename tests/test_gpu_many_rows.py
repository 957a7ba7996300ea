"""The row buckets' scan over many tiles of 1024 rows (k_scan_tiles, k_scan_sums), and row sorts in more than
one round of workgroups, where rows go 16 by 16: list order by the injection's bits, and time."""
import numpy as np
import pytest

from fastbarnes import hip, interpolation
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


# rows around 16 tiles (loads in flight), 48 (beyond, k_scan_sums), 4096 (a round of it) and 512 * 1024 (rows 16
# by 16)
@pytest.mark.parametrize('rows', [8193, (1 << 14) - 1, 1 << 14, (1 << 14) + 1, (1 << 14) + 1025, 48 * 1024 - 1, 48 * 1024,
                                  48 * 1024 + 1, (1 << 19) - 1, (1 << 19) + 1, (1 << 19) + 40000, (1 << 22) - 1,
                                  (1 << 22) + 2050])
def test_many_rows_bitwise(orc, rows):
    rng = np.random.default_rng(rows)
    size, n = (5, rows), 20000
    y = np.concatenate([rng.uniform(0.0, rows - 1.001, n), rng.integers(0, rows - 1, 30).repeat(40) + 0.5,
                        np.full(700, rows - 1.5), np.full(30, 0.5)])
    pts = np.stack([rng.uniform(0.0, 3.999, len(y)), y], 1)
    val = rng.normal(0.0, 1.0, len(y)) * np.exp(rng.uniform(-10, 10, len(y)))
    vg, wg = np.zeros(size[::-1]), np.zeros(size[::-1])
    rv, rw = vg.copy(), wg.copy()
    interpolation._inject_data_2d(vg, wg, pts, val, np.zeros(2), np.ones(2), size)
    orc.inject_raw(rv, rw, pts, val, np.zeros(2), np.ones(2), size)
    assert np.array_equal(vg.view(np.uint64), rv.view(np.uint64))
    assert np.array_equal(wg.view(np.uint64), rw.view(np.uint64))


def _times(f, fields):
    rng = np.random.default_rng(1)
    pts = hip.DeviceArray.from_numpy(rng.uniform(0.0, 1.0, (f['n'] * fields, 2)) * np.asarray(f['size']))
    val = hip.DeviceArray.from_numpy(rng.normal(0.0, 1.0, f['n'] * fields))
    batch = BarnesBatch([f] * fields)
    out = hip.DeviceArray((batch.total_out,), np.float32)
    s = hip.Stream()
    batch.set_timing(True)
    best = {}
    for _ in range(8):
        batch.execute(pts.ptr, val.ptr, out.ptr, s.ptr)
        s.synchronize()
        for k, ms in batch.stage_times().items():
            best[k] = min(best.get(k, ms), ms)
    return best


def test_many_rows_time():
    """100 fields of 20000 rows and 8 points: the sort took 0.4 of the x pass."""
    best = _times(dict(sigma=5.0, x0=[0.0, 0.0], step=1.0, size=(16, 20000), n=8, num_iter=4, max_dist=3.5), 100)
    assert best['sort'] < 0.2 * best['pass_x']


# rows of fields of few points: 4096 and 8192 for 1024 threads, 2048 for 256; crowded rows (more than 64 points)
@pytest.mark.parametrize('rows,n', [(2048, 900), (2049, 900), (4096, 2049), (4097, 2048), (4097, 2049), (8192, 2048),
                                    (8192, 1), (8193, 500), (8191, 2000)])
@pytest.mark.parametrize('crowded', [False, True])
def test_few_points_of_many_rows_bitwise(orc, rows, n, crowded):
    rng = np.random.default_rng(rows + n)
    size = (9, rows)
    y = rng.uniform(0.0, rows - 1.001, n)
    if crowded:
        y[: n // 2] = rng.uniform(rows - 4.0, rows - 1.001, n // 2)
    pts, val = np.stack([rng.uniform(0.0, 7.999, n), y], 1), rng.normal(0.0, 1.0, n) * np.exp(rng.uniform(-9, 9, n))
    vg, wg = np.zeros(size[::-1]), np.zeros(size[::-1])
    rv, rw = vg.copy(), wg.copy()
    interpolation._inject_data_2d(vg, wg, pts, val, np.zeros(2), np.ones(2), size)
    orc.inject_raw(rv, rw, pts, val, np.zeros(2), np.ones(2), size)
    assert np.array_equal(vg.view(np.uint64), rv.view(np.uint64))
    assert np.array_equal(wg.view(np.uint64), rw.view(np.uint64))


def test_few_points_of_many_rows_time():
    """40 fields of 5000 rows and 8 points: the sort took 0.48 of the x pass."""
    best = _times(dict(sigma=5.0, x0=[0.0, 0.0], step=1.0, size=(16, 5000), n=8, num_iter=4, max_dist=3.5), 40)
    assert best['sort'] < 0.35 * best['pass_x']
