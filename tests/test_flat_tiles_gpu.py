"""Tiled 2-D projections (distance driven and separable footprint) against the
one-thread-per-output kernels (VIR_PER_OUTPUT), where tiles, bands and blocks
end.

The distance-driven forward adds the same float64 terms in another grouping:
equal to the last float32 digit, bar 1e-7 relative L2.  The others form
overlaps from the same float32 intervals; backward in bins from the detector's
centre, where a boundary rounds by at most 3 * 2^-24 * nu / 2 (nu <= 700: 6e-5
bin) per view, random in sign against data of spread 0.23: below 2e-5 /
sqrt(views) relative.  Bar 1e-5 for the 5 or more views here.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    dict(shape=(2, 3), nu=5, na=8),
    dict(shape=(16, 16), nu=127, na=9, du=0.3),
    dict(shape=(17, 31), nu=128, na=8, su=0.25),
    dict(shape=(33, 15), nu=129, na=70, su=-0.4),      # more views than a wave has lanes
    dict(shape=(300, 40), nu=60, na=7, du=3.0),        # a tile's band spans several stages
    dict(shape=(40, 300), nu=300, na=5, du=0.6),
    dict(shape=(70, 66), nu=700, na=8, du=0.15),       # pixels wider than three bins
    dict(shape=(500, 520), nu=700, na=6, du=1.1),      # tiles enough for four waves each
    dict(shape=(130, 65), nu=520, na=260, du=0.4),     # the same forward
]


def _make(kind, geom, c, batch):
    c = dict(c)
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    if geom != "par":
        R = 0.5 * np.hypot(*shape)
        c.update(DSO=2.2 * R, DSD=3.1 * R)
        if c.get("du", 1.0) * nu > 5.0 * R:   # keep the detector inside 45 degrees
            c["du"] = 5.0 * R / nu
    ang = np.arange(na) * (2 * np.pi / na)
    if kind == "dd":
        from vir_amd.sys_mat.dd import DDProjector
        return DDProjector(shape, ang, nu, "par" if geom == "par" else "fan",
                           detector="flat" if geom == "par" else geom, **c)
    from vir_amd.sys_mat.pd import SFProjector
    return SFProjector(shape, ang, nu, "par" if geom == "par" else "fan", batch=batch, **c)


def _per_output(P, kind, fp, x, shape):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    out = torch.empty(shape, device="cuda")
    name = ("vir_dd2d_" if kind == "dd" else "vir_sf_") + ("fp" if fp else "bp")
    trig = [_lib.ptr(P.cos), _lib.ptr(P.sin)]
    trig = trig if kind == "dd" else [_lib.ptr(P.ang)] + trig
    _lib.check(getattr(_lib.lib(), name)(P.g, *trig, _lib.ptr(x), _lib.ptr(out), P.fp_scale, _lib.VIR_PER_OUTPUT,
                                         stream()), name)
    return out


def _rel(a, b):
    a, b = a.double(), b.double()
    assert float(b.abs().max()) > 0
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("kind,geom", [("dd", "par"), ("dd", "flat"), ("dd", "arc"), ("sf", "par"), ("sf", "flat")])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_tiles_match_gather(k, kind, geom):
    import torch
    P = _make(kind, geom, CASES[k], 1 + k % 3)
    vshape = P.vol_shape if kind == "sf" else P.img_shape
    rng = np.random.default_rng(k)
    x = torch.from_numpy(rng.uniform(0.2, 1.0, vshape).astype(np.float32)).cuda()
    y = torch.from_numpy(rng.uniform(0.2, 1.0, P.sino_shape).astype(np.float32)).cuda()
    fx, by = P.fp(x), P.bp(y)
    assert _rel(fx, _per_output(P, kind, True, x, P.sino_shape)) <= (1e-7 if kind == "dd" else 1e-5)
    assert _rel(by, _per_output(P, kind, False, y, vshape)) <= 1e-5
    assert torch.equal(fx, P.fp(x)) and torch.equal(by, P.bp(y))
    assert torch.allclose(P.fp(x, out=fx.clone(), accumulate=True), 2 * fx, rtol=1e-6, atol=0)
    assert torch.allclose(P.bp(y, out=by.clone(), accumulate=True), 2 * by, rtol=1e-6, atol=0)


@pytest.mark.parametrize("kind,geom", [("dd", "arc"), ("sf", "flat")])
def test_infinite_values_stay_where_they_are(kind, geom):
    import torch
    P = _make(kind, geom, dict(shape=(47, 40), nu=129, na=70, su=-0.4), 1)
    x = torch.ones(P.img_shape, device="cuda")
    x[8, 13] = float("inf")
    y = torch.ones(P.sino_shape, device="cuda")
    y[3, 60] = float("inf")
    for fp, v, shape in ((True, x, P.sino_shape), (False, y, P.img_shape)):
        a = P.fp(v) if fp else P.bp(v)
        b = _per_output(P, kind, fp, v, shape)
        assert not torch.isnan(a).any() and torch.isinf(b).any()
        assert torch.equal(torch.isinf(a), torch.isinf(b))
