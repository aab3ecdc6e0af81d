"""Tiled FBP: the Toeplitz filter and the shared-geometry backprojection
against float64 evaluations in torch, at the sizes where tiles, chunks and
views end.  Positions, weights and sums are float64; what is left is the
rounding of the stored float32 values, 2^-24 per value: bar 1.2e-7 relative L2.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BAR = 1.2e-7


def _rel(a, b):
    a, b = a.double(), b.double()
    assert float(b.abs().max()) > 0
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("rows,nu", [(1, 1), (1, 2), (3, 255), (2, 256), (5, 257), (2, 511), (3, 513), (2, 1025),
                                     (1, 4096)])
@pytest.mark.parametrize("weighted", [False, True])
def test_filter(rows, nu, weighted):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    r = np.random.default_rng(nu)
    x, t, w = (torch.from_numpy(r.normal(size=s).astype(np.float32)).cuda() for s in ((rows, nu), nu, nu))
    out = torch.empty_like(x)
    _lib.check(_lib.lib().vir_fbp_filter(_lib.ptr(x), rows, nu, _lib.ptr(w) if weighted else None, _lib.ptr(t),
                                         _lib.ptr(out), stream()), "vir_fbp_filter")
    i = torch.arange(nu, device="cuda")
    T = t.double()[(i[:, None] - i[None, :]).abs()]
    assert _rel(out, (x * w if weighted else x).double() @ T) <= BAR


def _bp64(P, q, geom, DSO, c0, step):
    import torch
    nx, ny = P.img_shape
    x = (torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5 - nx / 2)[:, None]
    y = (torch.arange(ny, dtype=torch.float64, device="cuda") + 0.5 - ny / 2)[None, :]
    out = torch.zeros(nx, ny, dtype=torch.float64, device="cuda")
    for a in range(P.na):
        c, s = float(P.cos[a]), float(P.sin[a])
        p, o = -s * x + c * y, DSO - (c * x + s * y)
        if geom == "par":
            pos, w = p, 1.0
        elif geom == "flat":
            pos, w = DSO / o * p, (DSO / o) ** 2
        else:
            pos, w = torch.atan2(p, o), 1.0 / (o * o + p * p)
        tf = (pos - c0) / step
        j = torch.floor(tf)
        fr = tf - j
        ok = (j >= -1) & (j <= P.nu - 1)
        row = torch.nn.functional.pad(q[a].double(), (1, 1))
        j = (j.long() + 1).clamp(0, P.nu)
        out += ok * w * ((1 - fr) * row[j] + fr * row[j + 1])
    return out * P.scale


@pytest.mark.parametrize("geom", ["par", "flat", "arc"])
@pytest.mark.parametrize("shape,nu,na,DSO", [((1, 1), 4, 3, 30.0), ((16, 17), 25, 5, 40.0), ((33, 15), 60, 70, 900.0),
                                             ((50, 61), 1, 4, 300.0), ((515, 510), 700, 4, 1200.0)])
def test_backprojection(geom, shape, nu, na, DSO):
    """Equiangular detector: DSO 30 and 40 take the near-source path, 300 the
    longer series, 900 and 1200 the shorter one."""
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    from vir_amd.fbp import FBP
    DSO, DSD, du, su = np.float32(DSO), np.float32(1.4 * DSO), np.float32(1.3), np.float32(0.25)
    P = FBP(shape, np.arange(na) * (2 * np.pi / na) + 0.1, nu, "par" if geom == "par" else "fan", DSO=float(DSO),
            DSD=float(DSD), du=float(du), su=float(su), detector="flat" if geom == "par" else geom)
    q = torch.from_numpy(np.random.default_rng(nu).normal(size=(na, nu)).astype(np.float32)).cuda()
    out = torch.empty(shape, device="cuda")
    _lib.check(_lib.lib().vir_fbp_bp(P.g, _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(q), _lib.ptr(out), P.scale, 0,
                                     stream()), "vir_fbp_bp")
    f = 1.0 if geom == "par" else float(DSO) / float(DSD) if geom == "flat" else 1.0 / float(DSD)
    ref = _bp64(P, q, geom, float(DSO), float(du) * (0.5 - 0.5 * nu + float(su)) * f, float(du) * f)
    assert _rel(out, ref) <= BAR
    two = out.clone()
    _lib.check(_lib.lib().vir_fbp_bp(P.g, _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(q), _lib.ptr(two), P.scale,
                                     _lib.VIR_ACCUMULATE, stream()), "vir_fbp_bp")
    assert torch.allclose(two, 2 * out, rtol=1e-6, atol=0)
