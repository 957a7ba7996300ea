"""FP32C column passes of widths that float4 tiles cannot take (load_columns): remainders of the
workgroup's columns and of its rows, one column to a tile, lines shorter than a step, chunked lines.
Against the FP64 path within the library's bound for FP32C, RMSE 1e-5 on values of order 10, and the
same nodes masked but for those whose weight lies within float32 rounding of the threshold (at most 1
in 1000)."""
import numpy as np
import pytest

from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('size', [(13, 12), (17, 40), (34, 41), (35, 300), (37, 599), (33, 1001), (18, 1201), (21, 2399),
                                  (13, 4801), (12, 12, 13), (17, 33, 12), (15, 14, 150), (13, 12, 1201), (29, 601, 13)])
@pytest.mark.parametrize('n', [40, 400])
def test_columns(size, n):
    rng = np.random.default_rng(sum(size) + n)
    dim = len(size)
    pts = rng.uniform(-0.5, np.asarray(size) - 0.5, (n, dim))
    val = 10.0 + rng.normal(0.0, 2.0, n)
    field = dict(sigma=1.5, x0=np.zeros(dim), step=1.0, size=size, n=n, num_iter=4, max_dist=3.5)
    got, ref = (BarnesBatch([field], precision=p).interpolate([pts], [val])[0] for p in ('fp32c', 'fp64'))
    assert np.mean(np.isnan(got) != np.isnan(ref)) <= 1e-3
    ok = ~np.isnan(got) & ~np.isnan(ref)
    assert ok.any()
    assert np.sqrt(np.mean((got[ok].astype(np.float64) - ref[ok]) ** 2)) <= 1e-5
