"""Parallel 3-D footprint projections with bins two and a half pixels wide and
more, on both sides of the lines between the tile and the gather.

As in test_sf_matrix_gpu the two add the same products in float64 in another
grouping: bar 1e-7 relative L2.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    dict(shape=(40, 44, 64), nu=24, nv=64, na=90, du=2.6, batch=3),              # 46 blocks an item
    dict(shape=(40, 44, 64), nu=24, nv=64, na=100, du=2.6, batch=3),             # 50
    dict(shape=(64, 60, 66), nu=33, nv=66, na=97, du=2.75, su=0.3),
    dict(shape=(60, 70, 40), nu=36, nv=50, na=150, du=2.7, dv=0.8),   # rows with slab sums
    dict(shape=(60, 70, 40), nu=36, nv=50, na=150, du=2.76, sv=0.3),
    dict(shape=(130, 121, 64), nu=60, nv=64, na=397, du=3.2),                    # 400 blocks
    dict(shape=(130, 121, 60), nu=60, nv=60, na=397, du=3.2),                    # 375
    dict(shape=(130, 121, 60), nu=60, nv=60, na=337, du=3.2, batch=2),           # 319
    dict(shape=(130, 121, 64), nu=60, nv=64, na=397, du=3.3),
    dict(shape=(130, 121, 100), nu=60, nv=100, na=397, du=3.0, sv=-0.4, dv=0.9),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_wide_bins_match_gather(k):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    from vir_amd.sys_mat.pd import SFProjector
    c = dict(CASES[k])
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    P = SFProjector(shape, np.arange(na) * (np.pi / na), nu, "par3d", **c)
    x = torch.from_numpy(np.random.default_rng(k).uniform(0.2, 1.0, P.vol_shape).astype(np.float32)).cuda()
    a, b = P.fp(x), torch.empty(P.sino_shape, device="cuda")
    _lib.check(_lib.lib().vir_sf_fp(P.g, _lib.ptr(P.ang), _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(x), _lib.ptr(b),
                                    P.fp_scale, _lib.VIR_PER_OUTPUT, stream()), "vir_sf_fp")
    assert float(b.abs().max()) > 0
    assert float((a.double() - b.double()).norm() / b.double().norm()) <= 1e-7
