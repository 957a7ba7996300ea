"""The FP64 injection (k_inject_cells) against the oracle, bit for bit: base cells whose target
cells meet in every combination, the grid's first and last cells, crowded cells and empty rows, both
sorts, cleared grids and grids that hold sums."""
import numpy as np
import pytest

from fastbarnes import interpolation

pytestmark = pytest.mark.gpu

FN = {1: interpolation._inject_data_1d, 2: interpolation._inject_data_2d, 3: interpolation._inject_data_3d}


@pytest.mark.parametrize('size', [(2,), (40,), (2, 2), (7, 2), (2, 9), (33, 20), (2, 2, 2), (5, 3, 4), (17, 12, 9)])
@pytest.mark.parametrize('n,crowd', [(1, 0.0), (30, 0.0), (700, 0.5), (9000, 0.2)])
def test_inject_cells_bitwise(orc, size, n, crowd):
    dim = len(size)
    rng = np.random.default_rng(n + sum(size))
    step, x0 = np.full(dim, 0.5), np.full(dim, -1.0)
    # base cells anywhere from one below the grid to one past it, some of them exactly on nodes
    c = rng.uniform(-1.0, 1.0, (n, dim)) + rng.integers(0, np.asarray(size), (n, dim))
    c[rng.random(n) < 0.1] = np.floor(c[rng.random(n) < 0.1][:1]) if n > 50 else 0.0
    c[rng.random(n) < crowd] = np.minimum(np.asarray(size) - 1.5, 1.25)
    pts = x0 + c * step
    val = rng.normal(0.0, 1.0, n) * np.exp(rng.uniform(-10, 10, n))
    for start in (0.0, 1.0):
        vg = start * rng.normal(0.0, 1.0, size[::-1])
        wg = start * rng.random(size[::-1])
        rv, rw = vg.copy(), wg.copy()
        FN[dim](vg, wg, pts, val, x0, step, size)
        orc.inject_raw(rv, rw, pts, val, x0, step, size)
        assert np.array_equal(vg.view(np.uint64), rv.view(np.uint64))
        assert np.array_equal(wg.view(np.uint64), rw.view(np.uint64))


@pytest.mark.parametrize('precision_n', [500, 9000])
def test_inject_cells_of_a_batch(orc, precision_n):
    """Several fields in one list (the cleared grids of a plan), with points outside each."""
    from fastbarnes.batched import BarnesBatch
    rng = np.random.default_rng(precision_n)
    fs = []
    for i, size in enumerate([(40, 30), (64, 17), (33, 33)]):
        n = [precision_n, 40, precision_n // 2][i]
        fs.append(dict(pts=rng.uniform(-0.5, np.asarray(size) * 0.25 + 0.5, (n, 2)), val=rng.normal(5.0, 2.0, n),
                       sigma=0.6, x0=np.zeros(2), step=0.25, size=size, num_iter=3, max_dist=3.5))
    batch = BarnesBatch([dict(sigma=c['sigma'], x0=c['x0'], step=c['step'], size=c['size'], n=len(c['val']),
                              num_iter=c['num_iter'], max_dist=c['max_dist']) for c in fs], precision='fp64')
    outs = batch.interpolate([c['pts'] for c in fs], [c['val'] for c in fs])
    for c, o in zip(fs, outs):
        ref = orc.interpolate_convol(c['pts'], c['val'], c['sigma'], c['x0'], c['step'], c['size'], num_iter=3,
                                     max_dist=3.5)
        ok = ~np.isnan(ref)
        assert np.array_equal(np.isnan(o), ~ok) and np.array_equal(o[ok].view(np.uint32), ref[ok].view(np.uint32))
