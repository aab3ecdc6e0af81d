"""Siddon projections whose rays are shared by several waves, and the walk of
rays in the plane, against the traced lists: every entry's float32 product is
summed in float64, so a ray's result is the lists' sum to one float32 rounding
(the order of float64 additions may move it by one unit); bar 1.2e-7 per ray.
Backprojection: float32 sums of at most a few hundred entries; bar 2e-6
relative L2 against float64.  Sizes on both sides of each rule (2, 4, 8 waves a
ray, small and large 2-D bricks), rays along axes, through corners and plane
intersections, from inside the grid, past it and tilted out of the plane."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sparse(src, trg, n, d, o):
    from vir_amd.sys_mat import siddon as sd
    ind, ln, off = sd.siddons(src, trg, n, d, o, flat=True)
    return ind, ln, np.repeat(np.arange(off.size - 1), np.diff(off))


def _check_fp(src, trg, n, d=1.0, o=0.0):
    import torch
    from vir_amd.sys_mat.siddon import SiddonProjector
    ind, ln, row = _sparse(src, trg, n, d, o)
    rng = np.random.default_rng(ind.size)
    vol = rng.uniform(0.2, 1.0, n).astype(np.float32)
    nrays = src.shape[0]
    ref = np.bincount(row, (vol.reshape(-1)[ind] * ln).astype(np.float64), nrays).astype(np.float32)
    x = torch.from_numpy(vol).cuda()
    for records in (True, False):
        P = SiddonProjector(src, trg, n, d, o, records=records)
        got = P.fp(x, check=True)
        err = np.abs(got.cpu().numpy().reshape(-1).astype(np.float64) - ref)
        assert (err <= 1.2e-7 * np.abs(ref)).all(), err.max()
        assert torch.equal(got, P.fp(x))
        assert torch.allclose(P.fp(x, out=got.clone(), accumulate=True), 2 * got, rtol=1e-6, atol=0)


def _scatter(m, seed, z, tilt=0.0):
    """m random segments in and around a 2-D grid of half width 10."""
    r = np.random.default_rng(seed)
    s, t = r.uniform(-16, 16, (2, m, 3))
    s[:, 2] = z
    t[:, 2] = z + tilt * r.uniform(-1, 1, m)
    k = max(m // 8, 1)
    s[:k, 0] = t[:k, 0]                                     # along y, some of them on a plane
    s[k:2 * k, 1] = t[k:2 * k, 1] = np.round(s[k:2 * k, 1])  # along x, on planes
    d = 16 * np.sign(r.uniform(-1, 1, k))
    s[2 * k:3 * k, :2] = np.stack([-d, -d], 1)              # through the corners of the voxels
    t[2 * k:3 * k, :2] = np.stack([d, d], 1)
    s[3 * k:4 * k, :2] *= 0.4                                # from inside
    return s.astype(np.float32), t.astype(np.float32)


@pytest.mark.parametrize("m", [1, 63, 64, 65, 700, 64 * 1024 + 5])
@pytest.mark.parametrize("z,tilt", [(0.0, 0.0), (0.3, 0.0), (0.0, 0.6)])
def test_flat_sets(m, z, tilt):
    s, t = _scatter(m, m, z, tilt)
    _check_fp(s, t, (20, 20, 1))


@pytest.mark.parametrize("n,d,o", [((17, 20, 1), 1.0, 0.25), ((13, 9, 1), 1.7, 0.0), ((1, 1, 1), 0.5, 0.0),
                                   ((40, 3, 1), (0.5, 2.0, 1.0), 0.0)])
def test_flat_grids(n, d, o):
    s, t = _scatter(300, 5, 0.1)
    _check_fp(s, t, n, d, o)


@pytest.mark.parametrize("m", [5, 900, 64 * 2048 + 1])
def test_solid_sets(m):
    r = np.random.default_rng(m)
    s, t = r.uniform(-14, 14, (2, m, 3)).astype(np.float32)
    s[: m // 4, 2] = t[: m // 4, 2]
    s[m // 4: m // 3, 0] = t[m // 4: m // 3, 0]
    _check_fp(s, t, (11, 16, 13))
    _check_fp(s, t, (16, 16, 16), 0.9)


@pytest.mark.parametrize("n,views,nu", [((33, 20, 1), 5, 50), ((128, 130, 1), 9, 190), ((224, 250, 1), 6, 300),
                                        ((16, 16, 1), 1, 25)])
@pytest.mark.parametrize("geom", ["par", "fan"])
def test_flat_backprojection(n, views, nu, geom):
    import torch
    from vir_amd.proj_geom import geom_circular
    from vir_amd.sys_mat.siddon import SiddonProjector
    dets = np.arange(nu) - (nu - 1) / 2
    s, t = geom_circular(dets, np.linspace(0.1, 3.0, views), geom, src_iso=600.0, det_iso=300.0) if geom == "fan" \
        else geom_circular(dets, np.linspace(0.1, 3.0, views), "par")
    P = SiddonProjector(s, t, n)
    ind, ln, row = _sparse(np.asarray(s), np.asarray(t), n, 1.0, 0.0)
    y = np.random.default_rng(views).uniform(0.2, 1.0, views * nu).astype(np.float32)
    ref = np.bincount(ind, y[row].astype(np.float64) * ln, int(np.prod(n)))
    got = P.bp(torch.from_numpy(y).cuda().reshape(P.ray_shape))
    g = got.cpu().numpy().reshape(-1).astype(np.float64)
    assert np.linalg.norm(g - ref) <= 2e-6 * np.linalg.norm(ref)
    assert torch.equal(got, P.bp(torch.from_numpy(y).cuda().reshape(P.ray_shape)))
