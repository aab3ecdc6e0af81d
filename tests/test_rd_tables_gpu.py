"""Ray-driven backprojection from LDS ray tables against the per-voxel gather
(VIR_PER_OUTPUT), at the sizes where bricks, tables and tiles end.

Both sum the same samples (path lengths) of the same float32 rays; their
weights differ by the rounding of positions, at most about 1.5 ulp of the
source distance (here <= 150 voxels: 1.3e-5 voxel) per sample, random in
sign.  A voxel's 16 samples of a view sum to weight 2, so the relative
difference is below 1.2e-5 / sqrt(views): bar 1e-5 relative L2.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CONE = [
    dict(shape=(2, 2, 2), nu=9, nv=9, na=4),
    dict(shape=(5, 9, 63), nu=40, nv=90, na=7),
    dict(shape=(13, 4, 64), nu=41, nv=93, na=6, su=0.3, sv=-0.4),
    dict(shape=(4, 17, 65), nu=38, nv=60, na=5, dv=1.7),
    dict(shape=(9, 10, 70), nu=150, nv=420, na=4, du=0.3, dv=0.3),   # tables overflow along u and v
    dict(shape=(8, 6, 30), nu=20, nv=700, na=4, dv=0.05),             # rows alone overflow a table
    dict(shape=(128, 125, 9), nu=140, nv=24, na=4, sv=58.0, DSO=120.0, DSD=180.0),  # four columns a wave
]
FLAT = [
    dict(shape=(2, 2), nu=7, na=1),
    dict(shape=(16, 8), nu=31, na=5),
    dict(shape=(17, 9), nu=40, na=32, su=0.25),
    dict(shape=(31, 23), nu=300, na=7, du=0.2),    # a tile meets more than 32 rays
    dict(shape=(500, 259), nu=700, na=3, DSO=400.0, DSD=600.0, bar=3e-5),  # tiles enough for four waves each
]


def _both(P, y):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    new = P.bp(y)
    old = torch.empty_like(new)
    _lib.check(_lib.lib().vir_rd_bp(P.g, _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(y), _lib.ptr(old), 1.0,
                                    _lib.VIR_PER_OUTPUT, stream()), "vir_rd_bp")
    assert torch.equal(new, P.bp(y))
    a, b = new.double().cpu().numpy(), old.double().cpu().numpy()
    assert np.abs(b).max() > 0
    acc = P.bp(y, out=new.clone(), accumulate=True)
    assert torch.allclose(acc, 2 * new, rtol=1e-6, atol=0)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _sino(shape, seed):
    import torch
    y = np.random.default_rng(seed).uniform(0.5, 1.5, shape).astype(np.float32)
    y.reshape(-1)[::11] = 0.0
    return torch.from_numpy(y).cuda()


@pytest.mark.parametrize("joseph", [False, True])
@pytest.mark.parametrize("k", range(len(CONE)))
def test_cone(k, joseph):
    from vir_amd.sys_mat.rd import RDProjector
    c = dict(CONE[k])
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    c.setdefault("DSO", 60.0)
    c.setdefault("DSD", 110.0)
    P = RDProjector(shape, np.arange(na) * (2 * np.pi / na), nu, "cone", d_pix=1.0, joseph=joseph, **c)
    assert _both(P, _sino(P.sino_shape, k)) <= 1e-5


@pytest.mark.parametrize("geom", ["par", "fan"])
@pytest.mark.parametrize("joseph", [False, True])
@pytest.mark.parametrize("k", range(len(FLAT)))
def test_flat(k, joseph, geom):
    from vir_amd.sys_mat.rd import RDProjector
    c = dict(FLAT[k])
    shape, nu, na, bar = c.pop("shape"), c.pop("nu"), c.pop("na"), c.pop("bar", 1e-5)
    if geom == "fan":
        c.setdefault("DSO", 60.0)
        c.setdefault("DSD", 90.0)
    else:
        c.pop("DSO", None)
        c.pop("DSD", None)
    P = RDProjector(shape, np.arange(na) * (2 * np.pi / na), nu, geom, d_pix=0.9, joseph=joseph, **c)
    assert _both(P, _sino(P.sino_shape, k)) <= bar
