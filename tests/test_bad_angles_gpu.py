"""A view without a finite angle takes part in nothing: its projection is zero
and it adds nothing to a backprojection, as in the one-thread-per-output kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEEP = [0, 1, 2, 3, 5, 6, 7]


def _angles(bad):
    a = np.arange(9) * 0.3
    a[[4, 8]] = bad
    return a


def _check_bp(P, Q, seed):
    import torch
    y = torch.rand(P.sino_shape, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))
    a, b = P.bp(y), Q.bp(y[KEEP].contiguous())
    # the same terms; float64 sums in other chains, one rounding of the result
    assert float((a - b).double().norm() / b.double().norm()) <= 1.2e-7


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("geom,joseph", [("par", False), ("par", True), ("fan", False), ("fan", True), ("cone", False),
                                         ("cone", True)])
def test_ray_driven(geom, joseph, bad):
    from vir_amd.sys_mat.rd import RDProjector
    shape, kw = ((40, 41, 6), dict(nv=7, sv=31.0)) if geom == "cone" else ((40, 41), {})
    if geom != "par":
        kw.update(DSO=140.0, DSD=210.0, du=1.5)
    P, Q = (RDProjector(shape, a, 70, geom, joseph=joseph, **kw) for a in (_angles(bad), _angles(0.0)[KEEP]))
    _check_bp(P, Q, 2)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("kind,geom", [("dd", "par"), ("dd", "flat"), ("dd", "arc"), ("dd", "cone"), ("sf", "par"),
                                       ("sf", "fan"), ("sf", "cone"), ("sf", "par3d"), ("sf", "par3d rows")])
def test_footprints(kind, geom, bad):
    import torch
    from vir_amd.sys_mat.dd import DDProjector
    from vir_amd.sys_mat.pd import SFProjector
    shape, kw = (40, 41), {}
    if geom in ("cone", "par3d", "par3d rows"):
        shape, kw = (40, 41, 6), dict(nv=7 if geom == "cone" else 6)
    if geom == "par3d rows":
        kw.update(dv=0.9, sv=0.2)
    if geom in ("flat", "arc", "fan", "cone"):
        kw.update(DSO=140.0, DSD=210.0, du=1.5)
    if kind == "dd":
        if geom in ("flat", "arc"):
            kw["detector"] = geom
        make = lambda a: DDProjector(shape, a, 70, "fan" if geom in ("flat", "arc") else geom, **kw)
    else:
        make = lambda a: SFProjector(shape, a, 70, geom.split()[0], **kw)
    P, Q = make(_angles(bad)), make(_angles(0.0)[KEEP])
    x = torch.rand(shape, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    a, b = P.fp(x), Q.fp(x)
    assert torch.equal(a[KEEP], b) and not bool(a[[4, 8]].any())
    _check_bp(P, Q, 4)
