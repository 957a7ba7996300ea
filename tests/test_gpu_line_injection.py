"""The FP32C x pass's injection (LineInjection) where its runs, chunks and row ranges have their edges:
runs of one cell up to and past a wave, lines of 1 to 128 lanes, rows without points, first and last
rows, columns and planes.  Against the FP64 path within the library's bound for FP32C, RMSE 1e-5 on
values of order 10, and the same nodes masked but for those whose weight lies within float32 rounding
of the threshold (at most 1 in 1000)."""
import numpy as np
import pytest

from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


def _run(c, precision):
    return BarnesBatch([c['field']], precision=precision).interpolate([c['pts']], [c['val']])[0]


@pytest.mark.parametrize('size', [(15,), (700,), (16, 20), (38, 41), (75, 20), (160, 30), (610, 12), (1300, 14),
                                  (2500, 12), (30, 14, 16), (290, 12, 13), (1250, 12, 12)])
@pytest.mark.parametrize('crowd', [1, 2, 15, 16, 17, 63, 64, 65, 200])
def test_runs(size, crowd):
    rng = np.random.default_rng(crowd + sum(size))
    dim = len(size)
    top = np.asarray(size) - 2
    cells = [np.zeros(dim, int), top, top // 2, top // 2 + np.eye(dim, dtype=int)[0], top // 3]
    pts = np.concatenate([np.asarray(c) + rng.uniform(0.0, 0.999, (crowd, dim)) for c in cells]
                         + [rng.uniform(-0.5, np.asarray(size) - 0.5, (60, dim))])
    rng.shuffle(pts)
    val = 10.0 + rng.normal(0.0, 2.0, len(pts))
    c = dict(pts=pts, val=val, field=dict(sigma=1.5, x0=np.zeros(dim), step=1.0, size=size, n=len(val), num_iter=4,
                                          max_dist=3.5))
    got, ref = _run(c, 'fp32c'), _run(c, 'fp64')
    assert np.mean(np.isnan(got) != np.isnan(ref)) <= 1e-3
    ok = ~np.isnan(got) & ~np.isnan(ref)
    assert ok.any()
    assert np.sqrt(np.mean((got[ok].astype(np.float64) - ref[ok]) ** 2)) <= 1e-5
