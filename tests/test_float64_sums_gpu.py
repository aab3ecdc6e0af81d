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
