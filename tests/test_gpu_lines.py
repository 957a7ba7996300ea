"""FP64 line passes (k_exact_stream) against the oracle, bit for bit, at the sizes where its
blocks, rings and launches change: line lengths and half kernels around multiples of the 16-step
block, the shortest line a kernel allows, line counts around the 8 lines of a workgroup, more
iterations than one launch takes, kernels that leave the LDS room for a few iterations or none."""
import numpy as np
import pytest

from fastbarnes import _lib, interpolation

pytestmark = pytest.mark.gpu


def _lines(tail, nlines, length, rect, num_iter, alpha, x):
    out = np.empty_like(x)
    _lib.check(_lib.lib().fb_accumulate_lines(int(tail), _lib.FB_PREC_FP64, nlines, length, rect, num_iter,
                                              float(alpha), x.ctypes.data, out.ctypes.data, 0, None))
    return out


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


# (half kernel, line length): 2T+2 is the shortest line of a kernel of 2T+1 terms
SHAPES = [(0, 2), (0, 16), (1, 4), (1, 17), (7, 16), (7, 33), (8, 18), (8, 64), (14, 31), (15, 32), (15, 47),
          (16, 34), (16, 257), (17, 49), (31, 64), (32, 128), (47, 200), (170, 400), (300, 700), (600, 1300)]


@pytest.mark.parametrize('T,length', SHAPES)
@pytest.mark.parametrize('num_iter,nlines', [(1, 1), (3, 8), (4, 9), (8, 3), (9, 17)])
def test_lines_bitwise(orc, T, length, num_iter, nlines):
    rng = np.random.default_rng(T * 1000 + length + num_iter)
    x = rng.normal(0.0, 1.0, (nlines, length)) * np.exp(rng.uniform(-20, 20, (nlines, length)))
    x[rng.random((nlines, length)) < 0.4] = 0.0
    x[rng.random((nlines, length)) < 0.1] = -0.0
    rect, alpha = 2 * T + 1, 0.2083
    got = _lines(True, nlines, length, rect, num_iter, alpha, x)
    ref = np.stack([orc.accumulate_tail_array(r.copy(), rect, num_iter, alpha) for r in x])
    assert np.array_equal(_bits(got), _bits(ref))
    got = _lines(False, nlines, length, rect, num_iter, 0.0, x)
    ref = np.stack([orc.accumulate_array(r.copy(), rect, num_iter) for r in x])
    assert np.array_equal(_bits(got), _bits(ref))


@pytest.mark.parametrize('rect,length', [(2, 16), (16, 40), (34, 50), (33, 34)])
def test_even_kernels_bitwise(orc, rect, length):
    x = np.random.default_rng(rect).normal(0.0, 1.0, (5, length))
    got = _lines(False, 5, length, rect, 4, 0.0, x)
    ref = np.stack([orc.accumulate_array(r.copy(), rect, 4) for r in x])
    assert np.array_equal(_bits(got), _bits(ref))


@pytest.mark.parametrize('size,num_iter', [((33, 47), 4), ((16, 129), 9), ((35, 18, 51), 3), ((18, 35, 33), 8)])
def test_grid_axes_bitwise(orc, size, num_iter):
    """Every axis of a grid (rows, columns, planes), with the NaN mask."""
    dim = len(size)
    rng = np.random.default_rng(sum(size))
    vg = rng.normal(0.0, 1.0, size[::-1])
    wg = np.abs(rng.normal(0.0, 1.0, size[::-1]))
    sigma, step = np.full(dim, 1.2), np.full(dim, 0.35)
    ks = 2 * interpolation._get_half_kernel_size_opt(sigma, step, num_iter) + 1
    tv = interpolation._get_tail_value(sigma, step, num_iter)
    v, w = vg.copy(), wg.copy()
    fn = interpolation._convolve_tail_2d if dim == 2 else interpolation._convolve_tail_3d
    fn(v, w, sigma, step, size, ks, num_iter, tv, 0.5)
    rv, rw = vg.copy(), wg.copy()
    orc.convolve(True, rv, rw, sigma, step, size, ks, num_iter, tv, 0.5)
    assert np.array_equal(_bits(v), _bits(rv))
    assert np.array_equal(np.isnan(w), np.isnan(rw))
    ok = ~np.isnan(rw)
    assert np.array_equal(_bits(w[ok]), _bits(rw[ok]))


@pytest.mark.parametrize('sigma,num_iter', [(0.4, 5), (6.0, 1), (20.0, 1)])
def test_1d_field_bitwise(orc, sigma, num_iter):
    """The last axis along rows, whose kernel writes the quotient; at sigma 20 (T = 692) the rings
    do not fit the LDS and one thread walks each line."""
    rng = np.random.default_rng(3)
    pts, val = rng.uniform(-1.0, 101.0, 300), rng.normal(10.0, 1.0, 300)
    c = dict(sigma=sigma, x0=0.0, step=0.05, size=2001, num_iter=num_iter, max_dist=3.5)
    out = interpolation.barnes(pts, val, **c)
    ref = orc.interpolate_convol(pts, val, c['sigma'], c['x0'], c['step'], (c['size'],), num_iter=num_iter,
                                 max_dist=3.5)
    ref = np.asarray(ref[0] if isinstance(ref, tuple) else ref).reshape(out.shape)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(out[ok].view(np.uint32), ref[ok].view(np.uint32))
