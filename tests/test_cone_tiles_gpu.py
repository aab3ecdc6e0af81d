"""Tiled cone-beam projections (distance driven and separable footprint)
against the one-thread-per-output kernels (VIR_PER_OUTPUT), where tiles, lists
and slabs end.

Both evaluate the same weights in float32; the z overlaps are formed in units
of the cells instead of the detector, so a boundary differs by the rounding of
a coordinate of at most n/2 cells, 2^-24 * n/2 * 2 ~ 6e-6 cell for n = 100;
random in sign, over at least 8 lines a bin: relative L2 below 6e-6 * sqrt(2) /
sqrt(8) = 3e-6.  Bar 5e-6.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BAR = 5e-6

CASES = [
    dict(shape=(8, 9, 2), nu=15, nv=2, na=5),                        # fewer slabs than slots: the gather
    dict(shape=(9, 8, 3), nu=16, nv=3, na=4, dv=1.2),
    dict(shape=(16, 12, 63), nu=33, nv=63, na=8),                    # tile edges, axis and diagonal views
    dict(shape=(17, 30, 64), nu=17, nv=64, na=7, su=0.3, sv=-0.6),
    dict(shape=(24, 24, 65), nu=60, nv=129, na=8, dv=0.8),           # two slots
    dict(shape=(20, 21, 70), nu=47, nv=40, na=6, dv=4.5),            # four slots forward
    dict(shape=(20, 21, 20), nu=47, nv=150, na=6, dv=0.7, sv=0.25),  # four slots backward
    dict(shape=(40, 37, 11), nu=5, nv=17, na=5, du=21.0),            # bins wider than a list
    dict(shape=(70, 9, 12), nu=6, nv=30, na=5, du=40.0),             # and than the staged pixels
    dict(shape=(13, 11, 12), nu=300, nv=19, na=5, du=0.2),           # footprints wider than a list
]


def _pair(kind, c, batch=1):
    c = dict(c)
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    kw = dict(nv=c.pop("nv"), DSO=75.0, DSD=142.0, du=1.7, dv=1.9, d_pix=1.0)
    kw.update(c)
    ang = np.arange(na) * (2 * np.pi / na)
    if kind == "dd":
        from vir_amd.sys_mat.dd import DDProjector
        return DDProjector(shape, ang, nu, "cone", **kw)
    from vir_amd.sys_mat.pd import SFProjector
    return SFProjector(shape, ang, nu, "cone", batch=batch, **kw)


def _per_output(P, kind, fp, x, shape):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    out = torch.empty(shape, device="cuda")
    name = ("vir_ddcone_" if kind == "dd" else "vir_sf_") + ("fp" if fp else "bp")
    trig = [_lib.ptr(P.cos), _lib.ptr(P.sin)]
    trig = trig if kind == "dd" else [_lib.ptr(P.ang)] + trig
    _lib.check(getattr(_lib.lib(), name)(P.g, *trig, _lib.ptr(x), _lib.ptr(out), P.fp_scale, _lib.VIR_PER_OUTPUT,
                                         stream()), name)
    return out


def _rel(a, b):
    a, b = a.double(), b.double()
    assert float(b.abs().max()) > 0
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("kind", ["dd", "sf"])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_tiles_match_gather(k, kind):
    import torch
    P = _pair(kind, CASES[k], 1 + (k % 2 if kind == "sf" else 0))
    rng = np.random.default_rng(k)
    vshape = P.vol_shape if kind == "sf" else P.img_shape
    x = torch.from_numpy(rng.uniform(0.2, 1.0, vshape).astype(np.float32)).cuda()
    y = torch.from_numpy(rng.uniform(0.2, 1.0, P.sino_shape).astype(np.float32)).cuda()
    fx, by = P.fp(x), P.bp(y)
    assert _rel(fx, _per_output(P, kind, True, x, P.sino_shape)) <= BAR
    assert _rel(by, _per_output(P, kind, False, y, vshape)) <= BAR
    assert torch.equal(fx, P.fp(x)) and torch.equal(by, P.bp(y))
    assert torch.allclose(P.fp(x, out=fx.clone(), accumulate=True), 2 * fx, rtol=1e-6, atol=0)
    assert torch.allclose(P.bp(y, out=by.clone(), accumulate=True), 2 * by, rtol=1e-6, atol=0)


@pytest.mark.parametrize("kind", ["dd", "sf"])
def test_infinite_values_stay_where_they_are(kind):
    """An infinite voxel (bin) reaches the bins (voxels) it has weight on, and
    no value of zero weight next to it turns into NaN."""
    import torch
    P = _pair(kind, dict(shape=(17, 30, 64), nu=37, nv=64, na=7, su=0.3, sv=-0.6))
    x = torch.ones(P.img_shape, device="cuda")
    x[8, 13, 31] = float("inf")
    y = torch.ones(P.sino_shape, device="cuda")
    y[3, 17, 30] = float("inf")
    for fp, v, shape in ((True, x, P.sino_shape), (False, y, P.img_shape)):
        a = P.fp(v) if fp else P.bp(v)
        b = _per_output(P, kind, fp, v, shape)
        assert not torch.isnan(a).any() and torch.isinf(b).any()
        assert torch.equal(torch.isinf(a), torch.isinf(b))


@pytest.mark.parametrize("kind", ["dd", "sf"])
@pytest.mark.parametrize("k", [3, 4, 7, 8])
def test_infinite_and_nan_voxels_reach_only_their_bins(k, kind):
    """A voxel's value counts where its weight is not zero, and nowhere else:
    the bins a unit voxel projects on are the ones an infinite one spoils."""
    import torch
    P = _pair(kind, CASES[k])
    vshape = P.vol_shape if kind == "sf" else P.img_shape
    x = torch.from_numpy(np.random.default_rng(k).uniform(0.2, 1.0, vshape).astype(np.float32)).cuda()
    at = [x.numel() // 2 + 3, x.numel() // 3]
    ones, bad, none = torch.zeros_like(x), x.clone(), x.clone()
    ones.view(-1)[at] = 1.0
    none.view(-1)[at] = 0.0
    bad.view(-1)[at[0]] = float("inf")
    bad.view(-1)[at[1]] = float("nan")
    hit, got, ref = P.fp(ones) > 0, P.fp(bad), P.fp(none)
    assert hit.any() and not hit.all()
    assert torch.equal(~torch.isfinite(got), hit)
    # (without its voxel a sum's float64 additions group alike: one rounding)
    assert torch.allclose(got[~hit], ref[~hit], rtol=3e-7, atol=0)
