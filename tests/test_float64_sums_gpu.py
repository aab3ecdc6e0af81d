"""Sums of the footprint projectors are held in float64 from the first product on.

Geometries whose weights are exact (a view along an axis, power-of-two spacings
and scales): every product is exact or rounds once, so the result is the
correctly rounded sum, which a float32 partial sum misses in a good part of the
outputs.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(shape, seed):
    return np.random.default_rng(seed).uniform(0.2, 1.0, shape).astype(np.float32)


@pytest.mark.parametrize("kind", ["dd", "sf"])
@pytest.mark.parametrize("per,su", [(2, 0.5), (4, 0.5), (64, 0.0), (256, 0.5)])
def test_backprojection_over_many_bins(per, su, kind):
    """A pixel sums `per` bins a view; with an offset of half a bin its first
    and last count one half."""
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    from vir_amd.sys_mat.pd import SFProjector
    n, na = 6, 3
    P = (DDProjector if kind == "dd" else SFProjector)((5, n), np.zeros(na), n * per + 2, "par", du=1.0 / per, su=su)
    y = _values(P.sino_shape, per)
    w = np.ones(per + 1)
    w[0], w[-1] = (0.5, 0.5) if su else (1.0, 0.0)
    first = 0 if su else 1   # of pixel 0: the detector has a bin to spare at each end
    ref = sum((y[:, first + k:first + k + n * per:per].astype(np.float64) * w[k]).sum(0) for k in range(per + 1))
    out = P.bp(torch.from_numpy(y).cuda()).cpu().numpy()
    assert np.array_equal(out, np.broadcast_to(ref.astype(np.float32), (5, n)))


def test_cone_rows_over_several_slabs():
    """One line of pixels at magnification 2, each on one bin; a row meets half
    a slab, a whole one and another half."""
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    n, nz, na = 24, 66, 2
    P = DDProjector((1, n, nz), np.zeros(na), n, "cone", nv=33, DSO=4096.0, DSD=8192.0, du=2.0, dv=4.0, sv=0.25)
    x = _values((1, n, nz), 1)
    zb = np.arange(nz + 1) - nz / 2.0
    vb = 2.0 * (np.arange(34) - 16.5 + 0.25)                 # row edges in slabs
    W = np.clip(np.minimum(zb[1:, None], vb[None, 1:]) - np.maximum(zb[:-1, None], vb[None, :-1]), 0.0, None)
    ref = x[0].astype(np.float64) @ W / 2.0                  # over the row's two slabs
    out = P.fp(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(out, np.broadcast_to(ref.astype(np.float32), (na, n, 33)))


def test_cone_slabs_over_several_rows():
    """The same line backprojected: a slab meets half a row, a whole one and
    another half."""
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    n, nz, na = 24, 40, 3
    P = DDProjector((1, n, nz), np.zeros(na), n, "cone", nv=82, DSO=4096.0, DSD=8192.0, du=2.0, dv=1.0, sv=0.5)
    y = _values(P.sino_shape, 2)
    zb = 2.0 * (np.arange(nz + 1) - nz / 2.0)                # slab edges in rows
    vb = np.arange(83) - 41.0 + 0.5
    W = np.clip(np.minimum(zb[1:, None], vb[None, 1:]) - np.maximum(zb[:-1, None], vb[None, :-1]), 0.0, None)
    ref = y.astype(np.float64).sum(0) @ W.T                  # (24, 82) x (82, 40)
    out = P.bp(torch.from_numpy(y).cuda()).cpu().numpy()
    assert np.array_equal(out, ref.astype(np.float32)[None])
