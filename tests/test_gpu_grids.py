"""Launches of 2^32 work-items and more, which run in parts: every part against launches that need no
second one, bit for bit."""
import ctypes

import numpy as np
import pytest

from fastbarnes import _lib
from fastbarnes.batched import BarnesBatch

pytestmark = pytest.mark.gpu


def _need(gib):
    import torch
    if torch.cuda.mem_get_info()[0] < gib << 30:
        pytest.skip('needs %d GiB of free device memory' % gib)
    return torch


def test_inject_cells_in_parts():
    """Just over 2^29 points of a 3D grid, 8 threads each, against the two halves of the points injected
    one after the other: the grids' contents are added to in point order either way."""
    torch = _need(90)
    size, n = (16, 2048, 1024), (1 << 29) + 4099
    g = torch.Generator(device='cuda').manual_seed(7)
    pts = torch.rand((n, 3), generator=g, device='cuda', dtype=torch.float64)
    pts *= torch.tensor([15.0, 2047.0, 1023.0], device='cuda', dtype=torch.float64)
    val = torch.rand(n, generator=g, device='cuda', dtype=torch.float64)
    grids = torch.zeros((4,) + size[::-1], device='cuda', dtype=torch.float64)
    three = lambda x: (ctypes.c_double * 3)(x, x, x)

    def inject(a, b, vg, wg):
        torch.cuda.synchronize()
        _lib.check(_lib.lib().fb_inject(3, b - a, pts[a:b].data_ptr(), val[a:b].data_ptr(), three(0.0), three(1.0),
                                        (ctypes.c_int64 * 3)(*size), vg.data_ptr(), wg.data_ptr(),
                                        _lib.FB_FLAG_DEVICE_PTRS, None))

    inject(0, n, grids[0], grids[1])
    inject(0, n // 2, grids[2], grids[3])
    inject(n // 2, n, grids[2], grids[3])
    assert abs(grids[1].sum().item() / n - 1.0) < 1e-9
    assert torch.equal(grids[:2].view(torch.int64), grids[2:].view(torch.int64))


def test_fp64_lines_in_parts():
    """110 million x lines, 8 to a workgroup of 320 threads at 5 iterations, against the field's first
    rows and planes alone: the points' kernels end before either field does."""
    torch = _need(60)
    rng = np.random.default_rng(3)
    n = 4000
    val = torch.from_numpy(rng.normal(10.0, 2.0, n)).cuda()

    def run(size, pts):
        c = dict(sigma=1.2, x0=0.0, step=0.5, size=size, n=n, num_iter=5, max_dist=3.5)
        b = BarnesBatch([c], precision='fp64')
        out = torch.empty(b.total_out, device='cuda')
        torch.cuda.synchronize()
        s = torch.cuda.Stream()
        b.execute(pts.data_ptr(), val.data_ptr(), out.data_ptr(), s.cuda_stream)
        s.synchronize()
        return out.reshape(size[::-1])

    # (20 nodes and more from the lines' first ones, where a field ends and the other does not)
    corner = torch.from_numpy(rng.uniform(0.0, 1.0, (n, 3)) * [4.5, 20.0, 10.0] + [0.0, 10.0, 10.0]).cuda()
    small, big = (10, 150, 140), (10, 11000, 10000)
    ref, out = run(small, corner), run(big, corner)
    assert torch.equal(out[:100, :100].view(torch.int32), ref[:100, :100].view(torch.int32))
    assert int((~torch.isnan(out)).sum()) == int((~torch.isnan(ref)).sum()) > 0
    del out
    # the same points 10900 and 9900 nodes further on, among the last lines: their positions round
    # differently, so a weight may move across the threshold and values by float32 rounding
    far = corner + 0.5 * torch.tensor([0.0, 10900.0, 9900.0], device='cuda', dtype=torch.float64)
    out = run(big, far)[9900:, 10900:]
    ref = ref[:100, :100]
    assert (torch.isnan(out) != torch.isnan(ref)).float().mean() < 1e-4
    ok = ~torch.isnan(out) & ~torch.isnan(ref)
    assert torch.allclose(out[ok], ref[ok], rtol=1e-5)
