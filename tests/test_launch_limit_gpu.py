"""Calls whose tiles need more threads than one launch can have (2^32 - 1):
many small items, many short rows.  The result of a part is that of the part
alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NB = 17_000_000


def _same(P_many, P_one, fp, x):
    import torch
    a = P_many.fp(x) if fp else P_many.bp(x)
    for j in (0, 1, NB // 2, 16_777_214, 16_777_215, 16_777_216, NB - 1):
        one = P_one.fp(x[j].contiguous()) if fp else P_one.bp(x[j].contiguous())
        assert torch.equal(a[j], one), j
    assert bool(((a > 0) == (a[0] > 0)).all())


@pytest.mark.parametrize("geom,shape,nu,kw", [
    ("par", (2, 2), 2, {}),
    ("fan", (2, 2), 2, dict(DSO=9.0, DSD=12.0)),
    ("par3d", (2, 1, 6), 4, dict(nv=6)),
    ("cone", (1, 1, 3), 1, dict(nv=3, DSO=9.0, DSD=12.0, du=2.0)),
])
@pytest.mark.parametrize("fp", [True, False])
def test_many_small_items(geom, shape, nu, kw, fp):
    import torch
    from vir_amd.sys_mat.pd import SFProjector
    ang = np.array([0.3])
    many, one = (SFProjector(shape, ang, nu, geom, batch=b, **kw) for b in (NB, 1))
    n = many.vol_shape if fp else many.sino_shape
    x = torch.rand(n, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) + 0.5
    _same(many, one, fp, x)


def test_many_filtered_rows():
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    rows, nu = 11_300_000, 513
    if torch.cuda.mem_get_info()[0] < 60e9:
        pytest.skip("needs 46 GB of device memory")
    x = torch.empty(rows, nu, device="cuda").uniform_(0.5, 1.5)
    out = torch.zeros(rows, nu, device="cuda")
    t = torch.rand(nu, device="cuda")
    _lib.check(_lib.lib().vir_fbp_filter(_lib.ptr(x), rows, nu, None, _lib.ptr(t), _lib.ptr(out), stream()), "filter")
    i = torch.arange(nu, device="cuda")
    T = t.double()[(i[:, None] - i[None, :]).abs()]
    for r in (0, rows // 2, 11_184_809, 11_184_810, 11_184_811, rows - 1):
        ref = x[r].double() @ T
        assert float((out[r].double() - ref).norm() / ref.norm()) <= 1.2e-7
    assert float(out.min()) > 0
    del x, out
    torch.cuda.empty_cache()
