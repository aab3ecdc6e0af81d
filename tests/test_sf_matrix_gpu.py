"""Parallel 3-D separable footprint on the matrix cores against the
one-thread-per-output kernels (VIR_PER_OUTPUT): the same float32 weights and
values, multiplied exactly and summed in float64 in another grouping, so equal
to the last float32 digit of the result; bar 1e-7 relative L2.  Sizes where
pixel blocks, slab groups, view groups and bin windows end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BAR = 1e-7

CASES = [
    dict(shape=(1, 1, 1), nu=8, nv=1, na=1),
    dict(shape=(5, 7, 17), nu=16, nv=17, na=3, su=0.25),
    dict(shape=(8, 4, 64), nu=20, nv=64, na=65, su=-0.3),
    dict(shape=(9, 13, 65), nu=23, nv=65, na=8),
    dict(shape=(12, 11, 20), nu=25, nv=26, na=9),              # rows past both ends of the slabs
    dict(shape=(12, 11, 26), nu=25, nv=20, na=9, sv=2.0),      # slabs past the rows
    dict(shape=(10, 10, 33), nu=9, nv=33, na=260, du=4.0),     # one K-step
    dict(shape=(20, 18, 33), nu=50, nv=33, na=7, du=0.6),      # three
    dict(shape=(20, 18, 12), nu=70, nv=12, na=7, du=0.45),     # four
    dict(shape=(11, 9, 40), nu=30, nv=40, na=12, d_pix=0.7, dv=0.7, du=0.8),
    dict(shape=(256, 255, 3), nu=370, nv=3, na=5, batch=2),    # a wave a block
    dict(shape=(150, 20, 70), nu=100, nv=70, na=6),            # a narrow detector
    dict(shape=(20, 90, 7), nu=140, nv=7, na=260),             # many blocks an item: one wave group
    dict(shape=(20, 90, 7), nu=140, nv=7, na=260, sv=0.3),
    dict(shape=(50, 47, 40), nu=40, nv=67, na=22, sv=0.4, dv=0.6, du=2.3, batch=2),  # chunks of a line
    dict(shape=(50, 47, 8), nu=140, nv=8, na=22, du=0.4),
]


def _make(c):
    from vir_amd.sys_mat.pd import SFProjector
    c = dict(c)
    shape, nu, na = c.pop("shape"), c.pop("nu"), c.pop("na")
    return SFProjector(shape, np.arange(na) * (np.pi / na), nu, "par3d", **c)


def _per_output(P, fp, x, shape):
    import torch
    from vir_amd import _lib
    from vir_amd.device import stream
    out = torch.empty(shape, device="cuda")
    name = "vir_sf_fp" if fp else "vir_sf_bp"
    _lib.check(getattr(_lib.lib(), name)(P.g, _lib.ptr(P.ang), _lib.ptr(P.cos), _lib.ptr(P.sin), _lib.ptr(x),
                                         _lib.ptr(out), P.fp_scale, _lib.VIR_PER_OUTPUT, stream()), name)
    return out


@pytest.mark.parametrize("k", range(len(CASES)))
@pytest.mark.parametrize("fp", [False, True])
def test_matches_gather(k, fp):
    import torch
    P = _make(CASES[k])
    shape = (P.vol_shape, P.sino_shape) if fp else (P.sino_shape, P.vol_shape)
    x = torch.from_numpy(np.random.default_rng(k).uniform(0.2, 1.0, shape[0]).astype(np.float32)).cuda()
    f = P.fp if fp else P.bp
    a, b = f(x), _per_output(P, fp, x, shape[1])
    assert float(b.abs().max()) > 0
    assert float((a.double() - b.double()).norm() / b.double().norm()) <= BAR
    assert torch.equal(a, f(x))
    assert torch.allclose(f(x, out=a.clone(), accumulate=True), 2 * a, rtol=1e-6, atol=0)


@pytest.mark.parametrize("k", [1, 4, 10])
@pytest.mark.parametrize("fp", [False, True])
def test_infinite_and_nan_values_stay_where_they_are(k, fp):
    import torch
    P = _make(CASES[k])
    shape = (P.vol_shape, P.sino_shape) if fp else (P.sino_shape, P.vol_shape)
    x = torch.rand(shape[0], device="cuda", generator=torch.Generator("cuda").manual_seed(k))
    x.view(-1)[x.numel() // 2 + 3] = float("inf")
    x.view(-1)[x.numel() // 3] = float("nan")
    a, b = (P.fp if fp else P.bp)(x), _per_output(P, fp, x, shape[1])
    assert torch.isinf(b).any() or torch.isnan(b).any()
    assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
    ok = torch.isfinite(b)
    assert torch.allclose(a[ok], b[ok], rtol=3e-7, atol=0)
