"""A volume's projections have the same bits alone and in a batch, also where
the batch has many times the blocks of one item.

The data cancel to about 2^-23 of their size (every view comes twice with
opposite sign, the second time one unit in the last place larger; every line of
pixels likewise, for the view along the axis), so that another grouping of the
float64 additions shows in the float32 results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ("par", dict(shape=(64, 60), nu=92, na=90), 70),
    ("fan", dict(shape=(64, 60), nu=92, na=90, DSO=140.0, DSD=210.0, du=1.5), 70),
    ("fan", dict(shape=(16, 16), nu=140, na=9, DSO=40.0, DSD=60.0, du=0.3), 5),
    ("par", dict(shape=(16, 24), nu=30, na=45), 100),                       # narrow detectors: per output in the batch
    ("fan", dict(shape=(20, 16), nu=17, na=45, DSO=50.0, DSD=75.0, du=3.0), 600),
    ("par3d", dict(shape=(64, 60, 40), nu=96, nv=40, na=13), 40),
    ("par3d", dict(shape=(64, 60, 10), nu=96, nv=7, na=13, dv=0.8, sv=0.1), 40),
    ("par3d", dict(shape=(40, 44, 16), nu=30, nv=16, na=9, du=2.6), 40),
    ("par3d", dict(shape=(40, 44, 4), nu=70, nv=4, na=9), 40),
    ("cone", dict(shape=(20, 24, 30), nu=40, nv=33, na=7, DSO=75.0, DSD=142.0, du=1.7, dv=1.9), 12),
    ("cone", dict(shape=(40, 44, 3), nu=40, nv=4, na=7, DSO=75.0, DSD=142.0, du=1.7, dv=1.9), 40),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_items_do_not_depend_on_the_batch(k):
    import torch
    from vir_amd.sys_mat.pd import SFProjector
    geom, c, nb = CASES[k]
    c = dict(c)
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    ang = np.arange(na) * (2 * np.pi / na)
    ang = np.concatenate([ang, ang])
    one, many = (SFProjector(shape, ang, nu, geom, batch=b, **c) for b in (1, nb))
    rng = np.random.default_rng(k)
    x = rng.uniform(0.2, 1.0, many.vol_shape).astype(np.float32)
    y = rng.uniform(0.2, 1.0, many.sino_shape).astype(np.float32)
    x[:, 1::2] = -np.nextafter(x[:, 0::2], np.float32(2))
    y[:, na:] = -np.nextafter(y[:, :na], np.float32(2))
    x, y = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    fx, by = many.fp(x), many.bp(y)
    for j in (0, nb // 2, nb - 1):
        assert torch.equal(fx[j], one.fp(x[j].contiguous())), (geom, "fp", j)
        assert torch.equal(by[j], one.bp(y[j].contiguous())), (geom, "bp", j)
