"""The sort of many small fields (k_field_sort of 256 threads): the same bits as each field alone, whose sort
takes 1024 threads, and as few rounds of workgroups as there are."""
import numpy as np
import pytest

from fastbarnes import hip
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


def _field(rng, size, n, hot):
    d = len(size)
    pts = rng.uniform(-0.02, 1.0, (n, d)) * np.asarray(size)
    if hot:   # more than 64 points of a bucket: the bitonic network
        pts[: n // 2] = rng.uniform(0.3, 0.7, (1, d)) * np.asarray(size)
    f = dict(sigma=3.0 if d < 3 else 1.5, x0=[0.0] * d, step=1.0, size=size, n=n, num_iter=4, max_dist=3.5)
    return f, pts, rng.normal(5.0, 2.0, n)


def _bits(a):
    return np.where(np.isnan(a), np.float32(0), a).view(np.uint32), np.isnan(a)


# points around the limits of a thread's share, rows around 2048 (2049: 1024 threads for every field)
@pytest.mark.parametrize('precision', ['fp32c', 'fp64'])
@pytest.mark.parametrize('size,n,hot', [((20, 30), 1, False), ((20, 30), 255, False), ((20, 30), 1024, False),
                                        ((20, 30), 1025, False), ((20, 30), 2048, False), ((20, 30), 2049, False),
                                        ((20, 30), 2047, True), ((300,), 900, True), ((300,), 2048, False),
                                        ((14, 2048), 700, False), ((14, 2049), 700, False),
                                        ((14, 13, 12), 1500, False), ((14, 13, 12), 300, True)])
def test_small_fields_bitwise(precision, size, n, hot):
    rng = np.random.default_rng(n)
    few = [_field(rng, size, n, hot) for _ in range(3)]
    fill = [_field(rng, tuple(min(s, 20) for s in size), 5, False) for _ in range(254)]
    run = lambda g: BarnesBatch([f for f, _, _ in g], precision=precision).interpolate([p for _, p, _ in g],
                                                                                       [v for _, _, v in g])
    got = run(few + fill)
    for k, g in enumerate(few):
        a, b = _bits(got[k]), _bits(run([g])[0])
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and not a[1].all()


def _sort_time(nf):
    rng = np.random.default_rng(nf)
    fields = [_field(rng, (30, 20), 50, False) for _ in range(nf)]
    pts = hip.DeviceArray.from_numpy(np.concatenate([p for _, p, _ in fields]))
    val = hip.DeviceArray.from_numpy(np.concatenate([v for _, _, v in fields]))
    batch = BarnesBatch([f for f, _, _ in fields])
    out = hip.DeviceArray((batch.total_out,), np.float32)
    s = hip.Stream()
    batch.set_timing(True)
    best = np.inf
    for _ in range(8):
        batch.execute(pts.ptr, val.ptr, out.ptr, s.ptr)
        s.synchronize()
        best = min(best, batch.stage_times()['sort'])
    return best


def test_small_fields_time():
    """2000 fields of 50 points: one after the other on a CU they took 4.8 times as long as 200."""
    assert _sort_time(2000) < 3.0 * _sort_time(200)
