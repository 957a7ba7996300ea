"""The row buckets' scan over many tiles of 1024 rows (k_scan_tiles, k_scan_sums), and row sorts in more than
one round of workgroups, where rows go 16 by 16: list order by the injection's bits, and time."""
import numpy as np
import pytest

from fastbarnes import hip, interpolation
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


# rows around 1, 2, 4096 and 4097 tiles (a round of k_scan_sums) and around 512 * 1024 (rows 16 by 16)
@pytest.mark.parametrize('rows', [8193, 1 << 14, (1 << 19) - 1, (1 << 19) + 1, (1 << 19) + 40000, (1 << 22) - 1,
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


def test_many_rows_time():
    """100 fields of 20000 rows and 8 points: the sort took 0.4 of the x pass."""
    rng = np.random.default_rng(1)
    f = dict(sigma=5.0, x0=[0.0, 0.0], step=1.0, size=(16, 20000), n=8, num_iter=4, max_dist=3.5)
    pts = hip.DeviceArray.from_numpy(rng.uniform(0.0, 1.0, (800, 2)) * np.asarray(f['size']))
    val = hip.DeviceArray.from_numpy(rng.normal(0.0, 1.0, 800))
    batch = BarnesBatch([f] * 100)
    out = hip.DeviceArray((batch.total_out,), np.float32)
    s = hip.Stream()
    batch.set_timing(True)
    best = {}
    for _ in range(8):
        batch.execute(pts.ptr, val.ptr, out.ptr, s.ptr)
        s.synchronize()
        for k, ms in batch.stage_times().items():
            best[k] = min(best.get(k, ms), ms)
    assert best['sort'] < 0.2 * best['pass_x']
