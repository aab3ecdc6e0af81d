"""TV denoising several iterations a pass (vir_tv_chambolle_pair) against the
two-launch iterations (vir_tv_chambolle): the same operations on every voxel,
so the same bits, where tiles, rows and chunks end and for every remainder of
the iterations."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 3), (17, 54), (16, 55), (40, 130), (300, 7), (1, 1, 1), (3, 2, 2), (8, 28, 60), (9, 29, 61),
          (30, 30, 64), (5, 57, 121), (70, 9, 65)]


def _run(shape, g, weight, iters, pair):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    from vir_amd.tv import TV_WORK
    nd = len(shape)
    dims = shape + (1,) * (3 - nd)
    q = torch.zeros((nd,) + shape, device="cuda")
    dmax = torch.full((TV_WORK,), 7.0, device="cuda")
    L, p, tau = _lib.lib(), _lib.ptr, 1.0 / (4 * nd)
    if pair:
        q2, cur = torch.full_like(q, float("nan")), ctypes.c_int32(0)
        _lib.check(L.vir_tv_chambolle_pair(nd, *dims, p(g), p(q), p(q2), ctypes.addressof(cur), weight, tau, iters,
                                           p(dmax), stream()), "pair")
        q = q2 if cur.value else q
    else:
        v = torch.empty_like(g)
        _lib.check(L.vir_tv_chambolle(nd, *dims, p(g), p(q), p(v), None, weight, tau, iters, p(dmax), stream()), "two")
    return q, dmax[:1].clone()


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("iters", [1, 2, 5, 8])
def test_same_bits(shape, iters):
    import torch
    rng = np.random.default_rng(len(shape) * 100 + iters)
    g = torch.from_numpy(rng.uniform(0, 1, shape).astype(np.float32)).cuda()
    a, da = _run(shape, g, 0.07, iters, True)
    b, db = _run(shape, g, 0.07, iters, False)
    assert torch.equal(a, b) and torch.equal(da, db)
    assert iters < 2 or max(shape) == 1 or float(a.abs().max()) > 0


def test_infinite_and_nan_voxels_spread_alike():
    import torch
    g = torch.rand(12, 40, 70, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    g[5, 20, 33] = float("inf")
    g[2, 29, 61] = float("nan")
    g[8, 3, 60] = 3e38
    a, _ = _run((12, 40, 70), g, 0.07, 4, True)
    b, _ = _run((12, 40, 70), g, 0.07, 4, False)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    ok = ~torch.isnan(b)
    assert torch.equal(a[ok], b[ok])
