"""Cone-beam projections of volumes and detectors a few slabs (rows) thick, on
both sides of the lines between the routes, against the one-thread-per-output
kernels.

Overlaps are formed in cells (rows) instead of detector units: as in
test_cone_tiles_gpu a boundary of n cells rounds by up to 2^-24 n / 2 * 2, here
below 6e-6 cell, random in sign over at least 8 views or lines: relative L2 below
3e-6.  Bar 5e-6.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BAR = 5e-6


def _per_output(P, name, x, shape):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    out = torch.empty(shape, device="cuda")
    trig = ([_lib.ptr(P.ang)] if name.startswith("vir_sf") else []) + [_lib.ptr(P.cos), _lib.ptr(P.sin)]
    _lib.check(getattr(_lib.lib(), name)(P.g, *trig, _lib.ptr(x), _lib.ptr(out), getattr(P, "fp_scale", 1.0),
                                         _lib.VIR_PER_OUTPUT, stream()), name)
    return out


def _rel(a, b):
    assert float(b.abs().max()) > 0
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("kind", ["dd", "sf"])
@pytest.mark.parametrize("nx,ny,nz,nv,batch", [
    (150, 149, 3, 3, 1), (150, 149, 5, 30, 1), (150, 149, 13, 12, 1), (150, 149, 18, 18, 1), (64, 66, 4, 5, 1),
    (130, 131, 66, 9, 1), (45, 40, 7, 6, 30),
])
def test_backprojection_of_thin_volumes(nx, ny, nz, nv, batch, kind):
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    from vir_amd.sys_mat.pd import SFProjector
    if batch > 1 and kind == "dd":
        pytest.skip("no batch")
    kw = dict(nv=nv, DSO=4.0 * nx, DSD=8.0 * nx, du=2.0, dv=2.0, su=0.25, sv=-0.2)
    ang = np.arange(9) * (2 * np.pi / 9)
    nu = int(1.3 * nx)
    P = DDProjector((nx, ny, nz), ang, nu, "cone", **kw) if kind == "dd" else \
        SFProjector((nx, ny, nz), ang, nu, "cone", batch=batch, **kw)
    y = torch.from_numpy(np.random.default_rng(nz).uniform(0.2, 1.0, P.sino_shape).astype(np.float32)).cuda()
    shape = P.img_shape if kind == "dd" else P.vol_shape
    a = P.bp(y)
    assert _rel(a, _per_output(P, "vir_ddcone_bp" if kind == "dd" else "vir_sf_bp", y, shape)) <= BAR
    assert torch.equal(a, P.bp(y))
    assert torch.allclose(P.bp(y, out=a.clone(), accumulate=True), 2 * a, rtol=1e-6, atol=0)


@pytest.mark.parametrize("kind", ["dd", "sf"])
def test_infinite_rows_of_thin_volumes(kind):
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    from vir_amd.sys_mat.pd import SFProjector
    P = (DDProjector if kind == "dd" else SFProjector)((150, 149, 5), np.arange(5) * 1.3, 200, "cone", nv=9, DSO=600.0,
                                                       DSD=1200.0, du=2.0, dv=2.0)
    y = torch.ones(P.sino_shape, device="cuda")
    y[2, 90, 4] = float("inf")
    y[3, 91, 3] = float("nan")
    a, b = P.bp(y), _per_output(P, "vir_ddcone_bp" if kind == "dd" else "vir_sf_bp", y, P.img_shape)
    assert torch.isinf(b).any() and torch.isnan(b).any()
    assert torch.equal(torch.isinf(a), torch.isinf(b)) and torch.equal(torch.isnan(a), torch.isnan(b))


@pytest.mark.parametrize("kind", ["dd", "sf"])
@pytest.mark.parametrize("nv,na,nu", [(3, 93, 400), (3, 92, 400), (4, 177, 400), (4, 176, 400), (5, 180, 400)])
def test_projection_onto_few_rows(nv, na, nu, kind):
    """25 blocks a view: 3 rows of 92 views and 4 of 176 are on the line."""
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    from vir_amd.sys_mat.pd import SFProjector
    n = 24
    P = (DDProjector if kind == "dd" else SFProjector)((n, n + 1, 7), np.arange(na) * (2 * np.pi / na), nu, "cone", nv=nv,
                                                       DSO=4.0 * n, DSD=8.0 * n, du=0.2, dv=2.0, sv=0.3)
    x = torch.from_numpy(np.random.default_rng(nv).uniform(0.2, 1.0, P.img_shape).astype(np.float32)).cuda()
    assert _rel(P.fp(x), _per_output(P, "vir_ddcone_fp" if kind == "dd" else "vir_sf_fp", x, P.sino_shape)) <= BAR


@pytest.mark.parametrize("joseph", [False, True])
@pytest.mark.parametrize("nx,ny,nz", [(104, 200, 2), (100, 200, 2), (160, 200, 3), (156, 200, 3), (160, 200, 2), (160, 199, 4)])
def test_ray_driven_backprojection_of_thin_volumes(nx, ny, nz, joseph):
    """26 x 25 and 40 x 25 bricks: 650 and 1000 are on the lines.  Joseph's samples
    are placed in voxel units here and along the ray there: a position of up to
    4 n = 800 voxels rounds by 2^-24 * 800 = 5e-5 voxel, against weights of order
    one, random over 7 views of a few rays each: bar 3e-5."""
    import torch
    from vir_amd.sys_mat.rd import RDProjector
    nu = 300
    P = RDProjector((nx, ny, nz), np.arange(7) * (2 * np.pi / 7), nu, "cone", nv=nz + 2, DSO=4.0 * ny, DSD=8.0 * ny, du=2.0,
                    dv=2.0, su=0.25, sv=(nu - nz - 2) / 2.0, joseph=joseph)
    y = torch.from_numpy(np.random.default_rng(nz).uniform(0.2, 1.0, P.sino_shape).astype(np.float32)).cuda()
    a = P.bp(y)
    assert _rel(a, _per_output(P, "vir_rd_bp", y, P.img_shape)) <= 3e-5
    assert torch.equal(a, P.bp(y))
