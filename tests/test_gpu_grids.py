"""Launches of 2^32 work-items and more, which run in parts: every part against launches that need no
second one, bit for bit."""
import ctypes

import pytest

from fastbarnes import _lib

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
