"""The work that users of this framework have it do, as measurable cases.

A case names an operation and its sizes.  `listed()` are fixed ones,
`draw(rng)` gives more of the same ranges, `prepare(case, seed)` makes what a
user's program holds before the call (measured data, a volume, the projector
object), `run(state)` is one pass through the public entry points, `work(case)`
the bytes and operations no implementation can avoid and `exact(case, seed)`
the outputs in float64 from plain torch, without this package.

Operations (all on data resident on the device, as iterative users keep it):

  siddon       one forward projection and the backprojection of its result,
               SiddonProjector on a circular orbit (2-D parallel or 3-D cone)
  siddon_sirt  a few SIRT iterations on a cone-beam Siddon projector, the
               serving loop's cone-beam job
  dd_sirt      a few SIRT iterations on the 2-D fan distance-driven pair, the
               serving loop's fan-beam job
  dd_cone      distance-driven cone-beam forward and backprojection
  sf_fan       separable-footprint fan-beam pair
  sf_cone      separable-footprint cone-beam pair
  sf_grad      one gradient step on 0.5 |Ax - b|^2 + lam TV(x) through
               torch.autograd, A the batched 3-D parallel footprint projector
  joseph_cone  ray-driven cone-beam pair, Joseph interpolation
  aw_fan       ray-driven fan-beam pair, Amanatides-Woo path lengths
  fbp          filtered backprojection (parallel, flat fan, equiangular fan)
  tv           total-variation denoising of an image or a volume, the step
               that SIRT + TV applies after each update
"""
import math

import numpy as np
import torch

DEV = "cuda"


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest reconstruction: 128^2, 180 parallel views, where launches and latency count
        dict(name="siddon_par_128", op="siddon", geom="par", nx=128, ny=128, nz=1, views=180, nu=185, nv=1),
        # a small served cone-beam job
        dict(name="siddon_sirt_cone_64", op="siddon_sirt", geom="cone", nx=64, ny=64, nz=64, views=120, nu=96, nv=96,
             iters=5),
        # the headline scan: 256^3, 360 views of a 512 x 384 detector
        dict(name="siddon_cone_256", op="siddon", geom="cone", nx=256, ny=256, nz=256, views=360, nu=512, nv=384),
        # the fan-beam SIRT benchmark: 512^2, 720 views, 888 equiangular bins
        dict(name="dd_sirt_fan_512", op="dd_sirt", geom="arc", nx=512, ny=512, nz=1, views=720, nu=888, nv=1, iters=3),
        # distance-driven cone beam at the middle size of the serving trace
        dict(name="dd_cone_128", op="dd_cone", geom="cone", nx=128, ny=128, nz=128, views=180, nu=192, nv=192),
        # footprint fan pair at an ordinary 2-D size
        dict(name="sf_fan_256", op="sf_fan", geom="fan", nx=256, ny=256, nz=1, views=360, nu=444, nv=1),
        # footprint cone pair on a ragged volume and detector
        dict(name="sf_cone_ragged", op="sf_cone", geom="cone", nx=120, ny=132, nz=101, views=150, nu=187, nv=150),
        # the differentiable-projector benchmark: 8 volumes of 256 x 256 x 64, 180 views
        dict(name="sf_grad_8x256", op="sf_grad", geom="par", batch=8, nx=256, ny=256, nz=64, views=180, nu=384, nv=64),
        # ray-driven cone pair, the interpolating option
        dict(name="joseph_cone_128", op="joseph_cone", geom="cone", nx=128, ny=128, nz=128, views=180, nu=192, nv=192),
        # a small ray-driven fan pair of odd sizes
        dict(name="aw_fan_129", op="aw_fan", geom="fan", nx=129, ny=127, nz=1, views=181, nu=223, nv=1),
        # FBP of the fan benchmark, SIRT's initial image
        dict(name="fbp_fan_512", op="fbp", geom="arc", nx=512, ny=512, nz=1, views=720, nu=888, nv=1, filter="hann"),
        # the TV step of SIRT + TV on the headline volume
        dict(name="tv_256", op="tv", geom="none", nx=256, ny=256, nz=256, weight=0.05, most=50),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["siddon", "siddon_sirt", "dd_sirt", "dd_cone", "sf_fan", "sf_cone", "sf_grad", "joseph_cone",
                     "aw_fan", "fbp", "tv"])
    if op == "tv":
        if rng.random() < 0.5:
            return dict(op=op, geom="none", nx=_log(rng, 128, 1024), ny=_log(rng, 128, 1024), nz=1,
                        weight=round(rng.uniform(0.02, 0.2), 3), most=rng.choice([20, 50, 100]))
        return dict(op=op, geom="none", nx=_log(rng, 48, 256), ny=_log(rng, 48, 256), nz=_log(rng, 48, 256),
                    weight=round(rng.uniform(0.02, 0.2), 3), most=rng.choice([20, 50]))
    if op in ("dd_sirt", "sf_fan", "aw_fan", "fbp") or (op == "siddon" and rng.random() < 0.5):
        n = _log(rng, 128, 1024 if op == "fbp" else 640)
        case = dict(op=op, geom="fan", nx=n, ny=n + rng.choice([0, 0, -5, 7]), nz=1, views=_log(rng, 90, 720),
                    nu=int(n * rng.uniform(1.45, 1.75)), nv=1)
        if op == "siddon":
            case["geom"] = "par"
        elif op == "dd_sirt":
            case.update(geom=rng.choice(["arc", "flat"]), iters=rng.choice([1, 2, 3]))
        elif op == "fbp":
            case.update(geom=rng.choice(["par", "flat", "arc"]), filter=rng.choice(["ramp", "hann", "shepp-logan"]))
        return case
    if op == "sf_grad":
        n = _log(rng, 96, 256)
        nz = _log(rng, 20, 80)
        return dict(op=op, geom="par", batch=rng.choice([1, 2, 3, 4, 8]), nx=n, ny=n + rng.choice([0, 3, -6]), nz=nz,
                    views=_log(rng, 45, 180), nu=int(n * rng.uniform(1.4, 1.6)), nv=nz)
    n = _log(rng, 48, 128 if op == "siddon_sirt" else 160)
    case = dict(op=op, geom="cone", nx=n, ny=n + rng.choice([0, 0, 9, -7]), nz=max(24, int(n * rng.uniform(0.6, 1.1))),
                views=_log(rng, 60, 240), nu=int(n * rng.uniform(1.3, 1.6)), nv=int(n * rng.uniform(1.1, 1.5)))
    if op == "siddon_sirt":
        case["iters"] = rng.choice([2, 3, 5])
    return case


# --------------------------------------------------------------- geometry

def _geo(case):
    """Distances, pitches, offsets (in bins) and view angles of a case: unit
    voxels; fan beam as the 512 / 720 / 888 benchmark scales with n; cone beam
    at magnification 2 as the serving jobs; a quarter-bin detector offset."""
    n = max(case["nx"], case["ny"])
    two_pi = 2 * np.pi if case["geom"] != "par" else np.pi
    ang = np.arange(case.get("views", 0)) * (two_pi / max(case.get("views", 0), 1))
    g = dict(d=1.0, du=1.0, dv=1.0, su=0.25, sv=0.0, DSO=0.0, DSD=0.0, ang=ang)
    if case["geom"] == "cone":
        g.update(DSO=4.0 * n, DSD=8.0 * n, du=2.0, dv=2.0)
        if case["nx"] == 256 and case["nu"] == 512:   # the headline scan: 0.5 mm voxels, 1 mm bins
            g.update(d=0.5, DSO=500.0, DSD=1000.0, du=1.0, dv=1.0)
    elif case["geom"] in ("fan", "flat", "arc"):
        DSO, DSD = 1000.0 * n / 512.0, 1500.0 * n / 512.0
        half = math.asin(n / math.sqrt(2.0) / DSO) * 1.02
        half = half if case["geom"] == "arc" else math.tan(half)
        g.update(DSO=DSO, DSD=DSD, du=2.0 * DSD * half / case["nu"])
    return g


def _bins(n, step, off):
    return step * (np.arange(n) - (n - 1) / 2.0 + off)


def _trig32(ang):
    """float32 cos and sin of float32 angles (what the 2-D and cone drivers
    define their views by), as float64 numbers."""
    a = np.asarray(ang, np.float32)
    return np.cos(a).astype(np.float64), np.sin(a).astype(np.float64)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _ellipses(seed, n_ell, ndim):
    r = np.random.default_rng(int(seed) + 1)
    cen = np.zeros((n_ell, 3))
    ax = np.ones((n_ell, 3))
    cen[:, :ndim] = r.uniform(-0.4, 0.4, (n_ell, ndim))
    ax[:, :ndim] = r.uniform(0.05, 0.45, (n_ell, ndim))
    th = r.uniform(0, np.pi, n_ell)
    rho = r.uniform(-0.2, 1.0, n_ell)
    rot = np.zeros((n_ell, 3, 3))
    for e in range(n_ell):
        c, s = np.cos(th[e]), np.sin(th[e])
        rot[e] = [[c, s, 0], [-s, c, 0], [0, 0, 1]]
    return cen, ax, rot, rho


def _phantom(shape, seed, n_ell=10):
    """Summed random ellipses (ellipsoids) in [-1, 1] per axis, float32."""
    ndim = 3 if len(shape) == 3 and shape[2] > 1 else 2
    dims = tuple(shape) if len(shape) == 3 else tuple(shape) + (1,)
    cen, ax, rot, rho = _ellipses(seed, n_ell, ndim)
    c = [((torch.arange(n, dtype=torch.float32, device=DEV) + 0.5) / n * 2 - 1) if n > 1 else
         torch.zeros(1, device=DEV) for n in dims]
    X, Y, Z = c[0][:, None, None], c[1][None, :, None], c[2][None, None, :]
    out = torch.zeros(dims, dtype=torch.float32, device=DEV)
    for e in range(n_ell):
        x, y, z = X - cen[e, 0], Y - cen[e, 1], Z - cen[e, 2]
        q = ((rot[e, 0, 0] * x + rot[e, 0, 1] * y) / ax[e, 0]) ** 2 + \
            ((rot[e, 1, 0] * x + rot[e, 1, 1] * y) / ax[e, 1]) ** 2 + (z / ax[e, 2]) ** 2
        out += (q <= 1.0) * float(rho[e])
    return out.reshape(shape).contiguous()


def _ray_points(case, g):
    """A point and a unit direction (float64) of every detector bin's ray, in
    detector order, for making measured data."""
    f64 = dict(dtype=torch.float64, device=DEV)
    c, s = (torch.tensor(v, **f64)[:, None, None] for v in (np.cos(g["ang"]), np.sin(g["ang"])))
    u = torch.tensor(_bins(case["nu"], g["du"], g["su"]), **f64)[None, :, None]
    v = torch.tensor(_bins(case["nv"], g["dv"], g["sv"]), **f64)[None, None, :]
    zero = torch.zeros(case["views"], case["nu"], case["nv"], **f64)
    if case["geom"] == "par":
        P = torch.stack([-s * u + zero, c * u + zero, v + zero], -1)
        h = torch.stack([c + zero, s + zero, zero], -1)
        return P, h
    P = torch.stack([g["DSO"] * c + zero, g["DSO"] * s + zero, zero], -1)
    if case["geom"] == "arc":
        a = u / g["DSD"]
        h = torch.stack([-c * torch.cos(a) - s * torch.sin(a) + zero, -s * torch.cos(a) + c * torch.sin(a) + zero,
                         zero], -1)
    else:
        h = torch.stack([-g["DSD"] * c - s * u + zero, -g["DSD"] * s + c * u + zero, v + zero], -1)
        h = h / h.norm(dim=-1, keepdim=True)
    return P, h


def _measured(case, g, seed, n_ell=8, noise=0.01):
    """Chord-length sinogram of the seed's ellipses with 1 % noise: measured
    data, not a projection of any pixel grid.  (views, nu[, nv]) float32."""
    P, h = _ray_points(case, g)
    half = torch.tensor([case["nx"], case["ny"], max(case["nz"], 2)], dtype=torch.float64, device=DEV) * (g["d"] / 2)
    cen, ax, rot, rho = _ellipses(seed, n_ell, 3 if case["nz"] > 1 else 2)
    b = torch.zeros(P.shape[:-1], dtype=torch.float64, device=DEV)
    for e in range(n_ell):
        R = torch.tensor(rot[e] / ax[e][:, None], dtype=torch.float64, device=DEV)
        q = (P / half - torch.tensor(cen[e], device=DEV)) @ R.T
        w = (h / half) @ R.T
        if case["nz"] == 1:
            q, w = q[..., :2], w[..., :2]
        ww, qw, qq = (w * w).sum(-1), (q * w).sum(-1), (q * q).sum(-1)
        b += float(rho[e]) * 2 * torch.sqrt((qw * qw - ww * (qq - 1)).clamp(min=0)) / ww
    b = b * (1 + noise * torch.randn(b.shape, dtype=torch.float64, device=DEV, generator=_gen(seed)))
    b = b.to(torch.float32)
    return b.contiguous() if case["nv"] > 1 or case["geom"] == "cone" else b[..., 0].contiguous()


def _shape(case):
    return (case["nx"], case["ny"], case["nz"]) if case["nz"] > 1 else (case["nx"], case["ny"])


def _inputs(case, seed):
    """The inputs of a case as plain tensors, made from the seed alone."""
    g, op = _geo(case), case["op"]
    if op == "tv":
        x = _phantom(_shape(case), seed)
        return g, x + 0.1 * torch.randn(x.shape, device=DEV, generator=_gen(seed))
    if op in ("siddon_sirt", "dd_sirt", "fbp"):
        return g, _measured(case, g, seed)
    if op == "sf_grad":
        shape = (case["nx"], case["ny"], case["nz"])
        vols = torch.stack([_phantom(shape, 100 * seed + k, 6) for k in range(case["batch"])])
        noisy = vols + 0.05 * torch.randn(vols.shape, device=DEV, generator=_gen(seed))
        b = torch.stack([_measured(dict(case), g, 100 * seed + k, 6) for k in range(case["batch"])])
        if case["batch"] == 1:
            noisy, b = noisy[0], b[0]
        return g, (noisy.contiguous(), b.contiguous())
    shape = (case["nx"], case["ny"], case["nz"]) if op == "siddon" else _shape(case)
    return g, _phantom(shape, seed)


# ------------------------------------------------------ prepare and run

LAM, EPS, RATE = 1e-3, 1e-2, 1e-5


def _siddon_projector(case, g):
    from vir_amd.geometry import circular_projections, circular_rays
    from vir_amd.sys_mat.siddon import SiddonProjector
    y = _bins(case["nu"], g["du"], g["su"])
    if case["geom"] == "par":
        args = (y, g["ang"], "par", 2.0 * case["nx"], 2.0 * case["nx"])
    else:
        args = (y, g["ang"], "cone", g["DSO"], g["DSD"] - g["DSO"], _bins(case["nv"], g["dv"], g["sv"]))
    src, trg = circular_rays(*args)
    return SiddonProjector(src, trg, (case["nx"], case["ny"], case["nz"]), g["d"], proj=circular_projections(*args))


def prepare(case, seed):
    op = case["op"]
    g, data = _inputs(case, seed)
    S = dict(op=op, case=case, data=data)
    det = {k: g[k] for k in ("du", "su", "DSO", "DSD")}
    det3 = {k: g[k] for k in ("du", "dv", "su", "sv", "DSO", "DSD")}
    if op in ("siddon", "siddon_sirt"):
        S["P"] = _siddon_projector(case, g)
    elif op == "dd_sirt":
        from vir_amd.sys_mat.dd import DDProjector
        S["P"] = DDProjector(_shape(case), g["ang"], case["nu"], "fan", detector=case["geom"], **det)
    elif op == "dd_cone":
        from vir_amd.sys_mat.dd import DDProjector
        S["P"] = DDProjector(_shape(case), g["ang"], case["nu"], "cone", nv=case["nv"], **det3)
    elif op == "sf_fan":
        from vir_amd.sys_mat.pd import SFProjector
        S["P"] = SFProjector(_shape(case), g["ang"], case["nu"], "fan", **det)
    elif op == "sf_cone":
        from vir_amd.sys_mat.pd import SFProjector
        S["P"] = SFProjector(_shape(case), g["ang"], case["nu"], "cone", nv=case["nv"], **det3)
    elif op == "sf_grad":
        from vir_amd.sys_mat.pd import SFProjector
        S["P"] = SFProjector((case["nx"], case["ny"], case["nz"]), g["ang"], case["nu"], "par3d", nv=case["nv"],
                             du=1.0, dv=1.0, su=g["su"], batch=case["batch"])
    elif op in ("joseph_cone", "aw_fan"):
        from vir_amd.sys_mat.rd import RDProjector
        if op == "aw_fan":
            S["P"] = RDProjector(_shape(case), g["ang"], case["nu"], "fan", **det)
        else:
            S["P"] = RDProjector(_shape(case), g["ang"], case["nu"], "cone", nv=case["nv"], joseph=True, **det3)
    elif op == "fbp":
        from vir_amd.fbp import FBP
        kw = dict(geom="par", du=g["du"], su=g["su"]) if case["geom"] == "par" else \
            dict(geom="fan", detector=case["geom"], **det)
        S["P"] = FBP(_shape(case), g["ang"], case["nu"], filter_type=case["filter"], **kw)
    if op in ("siddon_sirt", "dd_sirt"):
        # the normalisation sums, kept per geometry as the serving loop does
        P = S["P"]
        shape = (case["nx"], case["ny"], case["nz"]) if op == "siddon_sirt" else _shape(case)
        S["W_sino"] = P.fp(torch.ones(shape, device=DEV))
        S["W_img"] = P.bp(torch.ones_like(data))
    return S


def run(S):
    op, case = S["op"], S["case"]
    if op == "tv":
        from vir_amd.tv import denoise_tv_chambolle
        return denoise_tv_chambolle(S["data"], weight=case["weight"], max_num_iter=case["most"])
    P = S["P"]
    if op == "fbp":
        return P(S["data"])
    if op in ("siddon_sirt", "dd_sirt"):
        from vir_amd.sirt import SIRT
        return SIRT(P, S["data"], W_sino=S["W_sino"], W_img=S["W_img"]).run(case["iters"])
    if op == "sf_grad":
        from vir_amd.autograd import least_squares, project, total_variation
        x, b = S["data"]
        x = x.detach().requires_grad_(True)
        loss = least_squares(project(x, P), b) + LAM * total_variation(x, eps=EPS, ndim=3)
        (gx,) = torch.autograd.grad(loss, x)
        return {"loss": loss.detach().float(), "grad": gx, "x": x.detach() - RATE * gx}
    sino = P.fp(S["data"])
    return {"sino": sino, "back": P.bp(sino)}


# ------------------------------------------------------------------ work

def _entries(case):
    """(ray, voxel) or (bin, voxel) interactions of one projection, about."""
    nvox = case["nx"] * case["ny"] * case["nz"]
    bins = case["views"] * case["nu"] * case["nv"]
    op = case["op"]
    if op in ("siddon", "siddon_sirt"):   # crossings a ray, as the trace counts them
        return bins * case["nx"] * (0.88 if case["geom"] == "par" else 0.46)
    if op == "aw_fan":
        return bins * case["nx"] * 0.9
    if op == "joseph_cone":               # samples a ray, eight voxels each
        return bins * case["nx"] * 1.0 * 8
    if op in ("dd_sirt", "sf_fan"):
        return nvox * case["views"] * 2.3
    return nvox * case["views"] * 4.0     # about two bins along u and two along v


def work(case):
    op = case["op"]
    vol = 4.0 * case["nx"] * case["ny"] * case["nz"]
    if op == "tv":      # the image is read, the result written; the dual field is the method's own
        nd = 3 if case["nz"] > 1 else 2
        return {"bytes": 2 * vol, "flops": case["most"] * vol / 4 * 8 * nd}
    sino = 4.0 * case["views"] * case["nu"] * case["nv"]
    if op == "fbp":     # filtering by transforms, and one interpolation a pixel and view
        rows = case["views"] * case["nu"]
        return {"bytes": 2 * sino + sino + vol,
                "flops": rows * 10 * math.log2(2 * case["nu"]) + 8.0 * case["nx"] * case["ny"] * case["views"]}
    e = _entries(case)
    if op in ("siddon_sirt", "dd_sirt"):   # an iteration reads x, b, r and the weights and writes r and x
        return {"bytes": case["iters"] * (4 * sino + 4 * vol), "flops": case["iters"] * 4 * e}
    if op == "sf_grad":
        k = case["batch"]
        return {"bytes": k * (4 * vol + 3 * sino), "flops": k * (4 * e + 30 * vol / 4)}
    rays = 6 * sino if op == "siddon" else 0.0   # a ray set is given by its endpoints
    return {"bytes": 2 * (vol + sino + rays), "flops": 4 * e}


# ------------------------------------------------------------------ exact

F64 = torch.float64


def _t(a):
    return torch.as_tensor(np.asarray(a, np.float64), dtype=F64, device=DEV)


def _edges(n, d=1.0, off=0.0):
    return d * (torch.arange(n + 1, dtype=F64, device=DEV) - n / 2.0 + off)


class _Rows:
    """A sparse operator given view by view: `view(a)` yields (bins, pixels,
    weights), index tensors within the view's bins and the image."""

    def __init__(self, views, nbins, nvox, view, keep=False):
        self.na, self.nbins, self.nvox, self.view = views, nbins, nvox, view
        self.kept = [view(a) for a in range(views)] if keep else None

    def _parts(self, a):
        return self.kept[a] if self.kept is not None else self.view(a)

    def fp(self, x):
        y = torch.zeros(self.na, self.nbins, dtype=F64, device=DEV)
        x = x.reshape(-1).to(F64)
        for a in range(self.na):
            r, c, w = self._parts(a)
            y[a].index_add_(0, r, w * x[c])
        return y

    def bp(self, y):
        x = torch.zeros(self.nvox, dtype=F64, device=DEV)
        y = y.reshape(self.na, self.nbins).to(F64)
        for a in range(self.na):
            r, c, w = self._parts(a)
            x.index_add_(0, c, w * y[a][r])
        return x

    def pair(self, x):
        y = torch.zeros(self.na, self.nbins, dtype=F64, device=DEV)
        b = torch.zeros(self.nvox, dtype=F64, device=DEV)
        x = x.reshape(-1).to(F64)
        for a in range(self.na):
            r, c, w = self.view(a)
            y[a].index_add_(0, r, w * x[c])
            b.index_add_(0, c, w * y[a][r])
        return y, b


def _spread(lo, hi, edge0, step, n):
    """(interval index, bin, overlap) of intervals against n bins of width
    step from edge0, the positive overlaps."""
    lo, hi = lo.reshape(-1), hi.reshape(-1)
    j0 = torch.floor((lo - edge0) / step).long()
    span = int(torch.ceil((hi - lo).max() / step).item()) + 1
    I, J, W = [], [], []
    for t in range(span + 1):
        j = j0 + t
        e = edge0 + step * j
        ov = torch.minimum(hi, e + step) - torch.maximum(lo, e)
        ok = ((j >= 0) & (j < n) & (ov > 0)).nonzero().reshape(-1)
        I.append(ok)
        J.append(j[ok])
        W.append(ov[ok])
    return torch.cat(I), torch.cat(J), torch.cat(W)


def _trace(P, Q, n, d):
    """Voxels crossed by the segments P -> Q (R, 3) of a centred grid: (ray,
    voxel, length), by sorting the plane parameters."""
    D = Q - P
    L = D.norm(dim=1)
    al, lo, hi = [], torch.zeros(len(P), dtype=F64, device=DEV), torch.ones(len(P), dtype=F64, device=DEV)
    for a in range(3):
        pl = _edges(n[a], d)
        flat = D[:, a] == 0
        inv = 1.0 / torch.where(flat, torch.ones_like(D[:, a]), D[:, a])
        t = (pl[None, :] - P[:, a:a + 1]) * inv[:, None]
        t = torch.where(flat[:, None], torch.full_like(t, 2.0), t)
        t0, t1 = torch.minimum(t[:, 0], t[:, -1]), torch.maximum(t[:, 0], t[:, -1])
        inside = (P[:, a] >= pl[0]) & (P[:, a] <= pl[-1])
        lo = torch.where(flat, lo, torch.maximum(lo, t0))
        hi = torch.where(flat, torch.where(inside, hi, torch.full_like(hi, -1.0)), torch.minimum(hi, t1))
        al.append(t)
    t = torch.cat(al, 1)
    hi = torch.maximum(hi, lo)
    t = torch.minimum(torch.maximum(t, lo[:, None]), hi[:, None]).sort(dim=1).values
    dt, mid = t[:, 1:] - t[:, :-1], 0.5 * (t[:, 1:] + t[:, :-1])
    ray, k = (dt > 1e-13).nonzero(as_tuple=True)
    m = mid[ray, k]
    idx = [torch.floor((P[ray, a] + m * D[ray, a] + n[a] * d / 2.0) / d).long() for a in range(3)]
    ok = (idx[0] >= 0) & (idx[0] < n[0]) & (idx[1] >= 0) & (idx[1] < n[1]) & (idx[2] >= 0) & (idx[2] < n[2])
    vox = (idx[0] * n[1] + idx[1]) * n[2] + idx[2]
    return ray[ok], vox[ok], (dt[ray, k] * L[ray])[ok]


def _siddon_rows(case, g):
    """Rays as the reference's circular geometry lays them out: endpoints
    (-src, y), (det, y') rotated by the view angle, rounded to float32."""
    n = (case["nx"], case["ny"], case["nz"])
    y, z = _t(_bins(case["nu"], g["du"], g["su"])), _t(_bins(case["nv"], g["dv"], g["sv"]))
    src, det = (2.0 * n[0],) * 2 if case["geom"] == "par" else (g["DSO"], g["DSD"] - g["DSO"])

    def view(a):
        c, s = float(np.cos(g["ang"][a])), float(np.sin(g["ang"][a]))
        Y = y[:, None].expand(-1, len(z)).reshape(-1)
        Z = z[None, :].expand(len(y), -1).reshape(-1) if case["geom"] == "cone" else torch.zeros_like(Y)
        sy, sz = (Y, Z) if case["geom"] == "par" else (torch.zeros_like(Y), torch.zeros_like(Z))
        P = torch.stack([-src * c - sy * s, -src * s + sy * c, sz], 1).float().to(F64)
        Q = torch.stack([det * c - Y * s, det * s + Y * c, Z], 1).float().to(F64)
        return _trace(P, Q, n, g["d"])

    return _Rows(case["views"], case["nu"] * case["nv"], n[0] * n[1] * n[2], view)


def _sirt(A, b, iters):
    Ws = A.fp(torch.ones(A.nvox, dtype=F64, device=DEV)).reshape(-1)
    Wi = A.bp(torch.ones(A.na, A.nbins, dtype=F64, device=DEV))
    b, x = b.reshape(-1).to(F64), torch.zeros(A.nvox, dtype=F64, device=DEV)
    for _ in range(iters):
        r = A.fp(x).reshape(-1)
        r = torch.where(Ws != 0, (b - r) / torch.where(Ws != 0, Ws, torch.ones_like(Ws)), r)
        u = A.bp(r)
        x = x + torch.where(Wi != 0, u / torch.where(Wi != 0, Wi, torch.ones_like(Wi)), u)
    return x


def _drive(case, c, s):
    """Distance-driven lines of a view: driving axis x where |sin| >= |cos|."""
    xd = abs(np.float32(s)) >= abs(np.float32(c))
    if xd:
        return xd, case["nx"], case["ny"], -s, c, c, s, abs(s)
    return xd, case["ny"], case["nx"], c, -s, s, c, abs(c)


def _dd_fan_rows(case, g):
    C, S = _trig32(g["ang"])
    DSO, DSD, du, d = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du", "d"))
    u0 = du * (-case["nu"] / 2.0 + g["su"])

    def view(a):
        c, s = float(C[a]), float(S[a])
        xd, nd, no, pd, po, od, oo, rs = _drive(case, c, s)
        db, ob = _edges(nd, d)[None, :], _edges(no, d)
        oc = ((ob[:-1] + ob[1:]) / 2)[:, None]
        p, o = pd * db + po * oc, DSO - (od * db + oo * oc)
        pb = DSD * (torch.atan2(p, o) if case["geom"] == "arc" else p / o)
        den = DSO - oo * oc
        sc = torch.sqrt(den * den + (po * oc) ** 2) / (den * rs)
        i, j, w = _spread(torch.minimum(pb[:, :-1], pb[:, 1:]), torch.maximum(pb[:, :-1], pb[:, 1:]), u0, du, case["nu"])
        io, k = i // nd, i % nd
        return j, (k * case["ny"] + io) if xd else (io * case["ny"] + k), w * sc.reshape(-1)[io] * (d / du)

    # an iteration applies the operator four times: the entries are kept where they fit
    keep = case["views"] * case["nx"] * case["ny"] <= 2.2e8
    return _Rows(case["views"], case["nu"], case["nx"] * case["ny"], view, keep)


def _dd_cone_pair(case, g, x):
    C, S = _trig32(g["ang"])
    DSO, DSD, du, dv, d = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du", "dv", "d"))
    nx, ny, nz, nu, nv = (case[k] for k in ("nx", "ny", "nz", "nu", "nv"))
    u0, v0 = du * (-nu / 2.0 + g["su"]), dv * (-nv / 2.0 + g["sv"])
    vb = v0 + dv * torch.arange(nv + 1, dtype=F64, device=DEV)
    x = x.to(F64)
    sino = torch.zeros(case["views"], nu, nv, dtype=F64, device=DEV)
    back = torch.zeros_like(x)
    scale = d * d / (du * dv)
    for a in range(case["views"]):
        c, s = float(C[a]), float(S[a])
        xd, nd, no, pd, po, od, oo, rs = _drive(case, c, s)
        db, ob = _edges(nd, d)[None, :], _edges(no, d)
        oc = (ob[:-1] + ob[1:]) / 2
        pb = DSD * (pd * db + po * oc[:, None]) / (DSO - (od * db + oo * oc[:, None]))
        den = DSO - oo * oc
        sc = torch.sqrt(den * den + (po * oc) ** 2) / (den * rs)
        zb = (DSD / den)[:, None] * _edges(nz, d)[None, :]
        V = (torch.minimum(zb[:, 1:, None], vb[None, None, 1:]) -
             torch.maximum(zb[:, :-1, None], vb[None, None, :-1])).clamp(min=0)       # (no, nz, nv)
        X = (x.transpose(0, 1) if xd else x).contiguous()                              # (no, nd, nz)
        Y = torch.matmul(X, V).reshape(no * nd, nv)
        i, j, w = _spread(torch.minimum(pb[:, :-1], pb[:, 1:]), torch.maximum(pb[:, :-1], pb[:, 1:]), u0, du, nu)
        w = w * sc[i // nd] * scale
        sino[a].index_add_(0, j, w[:, None] * Y[i])
        B = torch.zeros(no * nd, nv, dtype=F64, device=DEV).index_add_(0, i, w[:, None] * sino[a][j])
        B = torch.matmul(B.reshape(no, nd, nv), V.transpose(1, 2).contiguous())
        back += B.transpose(0, 1) if xd else B
    return sino, back


def _sf_fan_rows(case, g):
    ang = np.asarray(g["ang"], np.float64)
    C, S = np.cos(ang).astype(np.float32).astype(np.float64), np.sin(ang).astype(np.float32).astype(np.float64)
    A = ang.astype(np.float32).astype(np.float64)
    DSO, DSD, du, d = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du", "d"))
    xb, yb = _edges(case["nx"], d)[:, None], _edges(case["ny"], d)[None, :]
    xc, yc = (xb[:-1] + xb[1:]) / 2, (yb[:, :-1] + yb[:, 1:]) / 2
    u0 = du * (-case["nu"] / 2.0 + g["su"])

    def view(a):
        c, s = float(C[a]), float(S[a])
        q = DSD * (-s * xb + c * yb) / (DSO - (c * xb + s * yb))
        q = torch.stack([q[:-1, :-1], q[1:, :-1], q[:-1, 1:], q[1:, 1:]])
        gam = torch.atan((-s * xc + c * yc) / (DSO - (c * xc + s * yc)))
        amp = 1.0 / (torch.cos(A[a] + gam).abs() + torch.sin(A[a] + gam).abs())
        i, j, w = _spread(q.amin(0), q.amax(0), u0, du, case["nu"])
        return j, i, w / du * amp.reshape(-1)[i] * d

    return _Rows(case["views"], case["nu"], case["nx"] * case["ny"], view)


def _sf_cone_pair(case, g, x):
    ang = np.asarray(g["ang"], np.float64)
    C, S = np.cos(ang).astype(np.float32).astype(np.float64), np.sin(ang).astype(np.float32).astype(np.float64)
    DSO, DSD, du, dv, d = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du", "dv", "d"))
    nx, ny, nz, nu, nv = (case[k] for k in ("nx", "ny", "nz", "nu", "nv"))
    xb, yb, zb = _edges(nx, d)[:, None], _edges(ny, d)[None, :], _edges(nz, d)
    xc, yc = (xb[:-1] + xb[1:]) / 2, (yb[:, :-1] + yb[:, 1:]) / 2
    u0, v0 = du * (-nu / 2.0 + g["su"]), dv * (-nv / 2.0 + g["sv"])
    X = x.to(F64).reshape(nx * ny, nz)
    sino = torch.zeros(case["views"], nu, nv, dtype=F64, device=DEV)
    back = torch.zeros(nx * ny * nz, dtype=F64, device=DEV)
    for a in range(case["views"]):
        c, s = float(C[a]), float(S[a])
        den = DSO - (c * xc + s * yc)
        uc, fm = DSD * (-s * xc + c * yc) / den, DSD / den
        q = -s * xb + c * yb
        q = fm * torch.stack([q[:-1, :-1], q[1:, :-1], q[:-1, 1:], q[1:, 1:]])
        cm = (fm / torch.cos(torch.atan(uc / DSD))).reshape(-1)
        amp = 1.0 / (abs(s) + abs(c))
        zz = cm[:, None] * zb[None, :]
        iv, m, wv = _spread(zz[:, :-1], zz[:, 1:], v0, dv, nv)
        pix = iv // nz
        wv = wv / dv
        Y = torch.zeros(nx * ny * nv, dtype=F64, device=DEV).index_add_(0, pix * nv + m, wv * X.reshape(-1)[iv])
        Y = Y.reshape(nx * ny, nv)
        i, j, wu = _spread(q.amin(0), q.amax(0), u0, du, nu)
        wu = wu / du * amp * d
        sino[a].index_add_(0, j, wu[:, None] * Y[i])
        B = torch.zeros(nx * ny, nv, dtype=F64, device=DEV).index_add_(0, i, wu[:, None] * sino[a][j])
        back.index_add_(0, iv, wv * B.reshape(-1)[pix * nv + m])
    return sino, back.reshape(nx, ny, nz)


def _sf_grad(case, g, data):
    x, b = data
    k, nx, ny, nz, nu, nv = (case[q] for q in ("batch", "nx", "ny", "nz", "nu", "nv"))
    ang = np.asarray(g["ang"], np.float64)
    C, S = np.cos(ang).astype(np.float32).astype(np.float64), np.sin(ang).astype(np.float32).astype(np.float64)
    xb, yb, zb = _edges(nx), _edges(ny), _edges(nz)
    xc, yc = ((xb[:-1] + xb[1:]) / 2)[:, None], ((yb[:-1] + yb[1:]) / 2)[None, :]
    u0 = -nu / 2.0 + g["su"]
    vb = _edges(nv)
    V = (torch.minimum(zb[1:, None], vb[None, 1:]) - torch.maximum(zb[:-1, None], vb[None, :-1])).clamp(min=0)
    X64 = x.to(F64).reshape(k, nx * ny, nz)
    X = torch.matmul(X64, V).transpose(0, 1).reshape(nx * ny, k * nv)
    B = b.to(F64).reshape(k, case["views"], nu, nv)
    G = torch.zeros(nx * ny, k * nv, dtype=F64, device=DEV)
    loss = 0.0
    for a in range(case["views"]):
        c, s = float(C[a]), float(S[a])
        w = abs(s) + abs(c)
        pc = -s * xc + c * yc
        i, j, wt = _spread(pc - 0.5 * w, pc + 0.5 * w, u0, 1.0, nu)
        wt = (wt / w)[:, None]
        r = torch.zeros(nu, k * nv, dtype=F64, device=DEV).index_add_(0, j, wt * X[i])
        r -= B[:, a].transpose(0, 1).reshape(nu, k * nv)
        loss += 0.5 * float((r * r).sum())
        G.index_add_(0, i, wt * r[j])
    G = torch.matmul(G.reshape(nx * ny, k, nv).transpose(0, 1), V.T.contiguous()).reshape(k, nx, ny, nz)
    X = X64.reshape(k, nx, ny, nz)
    D = [torch.zeros_like(X) for _ in range(3)]
    D[0][:, :-1] = X[:, 1:] - X[:, :-1]
    D[1][:, :, :-1] = X[:, :, 1:] - X[:, :, :-1]
    D[2][..., :-1] = X[..., 1:] - X[..., :-1]
    n = torch.sqrt(D[0] ** 2 + D[1] ** 2 + D[2] ** 2 + EPS * EPS)
    loss += LAM * float((n - EPS).sum())
    D = [q / n for q in D]
    T = -(D[0] + D[1] + D[2])
    T[:, 1:] += D[0][:, :-1]
    T[:, :, 1:] += D[1][:, :, :-1]
    T[..., 1:] += D[2][..., :-1]
    G = (G + LAM * T).reshape(x.shape)
    return {"loss": torch.tensor(loss, dtype=F64, device=DEV), "grad": G, "x": x.to(F64) - RATE * G}


def _aw_fan_rows(case, g):
    C, S = _trig32(g["ang"])
    DSO, DSD, du = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du"))
    u = _t(_bins(case["nu"], du, g["su"]))
    far = DSD + 2.0 * max(case["nx"], case["ny"])   # past the grid

    def view(a):
        c, s = float(C[a]), float(S[a])
        P = torch.tensor([DSO * c, DSO * s, 0.0], dtype=F64, device=DEV)
        h = torch.stack([-DSD * c - u * s, -DSD * s + u * c, torch.zeros_like(u)], 1)
        h = h / h.norm(dim=1, keepdim=True)
        return _trace(P.expand(len(u), 3), P + far * h, (case["nx"], case["ny"], 1), 1.0)

    return _Rows(case["views"], case["nu"], case["nx"] * case["ny"], view)


def _joseph_cone_pair(case, g, x):
    C, S = _trig32(g["ang"])
    DSO, DSD, du, dv = (float(np.float32(g[k])) for k in ("DSO", "DSD", "du", "dv"))
    n = (case["nx"], case["ny"], case["nz"])
    nu, nv = case["nu"], case["nv"]
    u = du * (torch.arange(nu, dtype=F64, device=DEV) - (nu / 2 - 0.5) + g["su"])
    v = dv * (torch.arange(nv, dtype=F64, device=DEV) - (nu / 2 - 0.5) + g["sv"])   # rows are centred with nu
    U, V = u[:, None].expand(nu, nv).reshape(-1), v[None, :].expand(nu, nv).reshape(-1)
    x = x.to(F64).reshape(-1)
    sino = torch.zeros(case["views"], nu * nv, dtype=F64, device=DEV)
    back = torch.zeros(n[0] * n[1] * n[2], dtype=F64, device=DEV)
    half = _t(n) / 2.0
    for a in range(case["views"]):
        c, s = float(C[a]), float(S[a])
        o = torch.tensor([DSO * c, DSO * s, 0.0], dtype=F64, device=DEV)
        h = torch.stack([-DSD * c - U * s, -DSD * s + U * c, V], 1)
        h = h / h.norm(dim=1, keepdim=True)
        hs = torch.where(h.abs() > 1e-6, h, torch.full_like(h, 1e-300))
        ta, tb = (-half - o) / hs, (half - o) / hs
        t0, t1 = torch.minimum(ta, tb).amax(1), torch.maximum(ta, tb).amin(1)
        hit = (t1 > t0).nonzero().reshape(-1)
        if not len(hit):
            continue
        K = int(((t1 - t0)[hit].max() / 0.5).item()) + 1
        for part in hit.split(max(1, 12_000_000 // K)):
            t = t0[part][:, None] + 0.5 * torch.arange(K, dtype=F64, device=DEV)[None, :]
            ray, k = (t <= t1[part][:, None]).nonzero(as_tuple=True)
            p = o + t[ray, k][:, None] * h[part[ray]] + (half - 0.5)
            ray = part[ray]
            for forward in (True, False):
                f0 = torch.trunc(p) if forward else torch.floor(p)
                dd, i0 = p - f0, f0.long()
                whole = (i0 >= 0).all(1) & (i0 < torch.tensor(n, device=DEV) - 1).all(1)
                for corner in range(8):
                    e = [(corner >> q) & 1 for q in range(3)]
                    idx = [i0[:, q] + e[q] for q in range(3)]
                    w = 0.5
                    for q in range(3):
                        w = w * (dd[:, q] if e[q] else 1 - dd[:, q])
                    ok = whole
                    if not forward:
                        ok = torch.ones_like(whole)
                        for q in range(3):
                            ok &= (idx[q] >= 0) & (idx[q] < n[q])
                    ok = ok.nonzero().reshape(-1)
                    vox = (idx[0][ok] * n[1] + idx[1][ok]) * n[2] + idx[2][ok]
                    if forward:
                        sino[a].index_add_(0, ray[ok], w[ok] * x[vox])
                    else:
                        back.index_add_(0, vox, w[ok] * sino[a][ray[ok]])
    return sino.reshape(-1, nu, nv), back.reshape(n)


def _fbp_exact(case, g, b):
    nu, du, su, DSO, DSD = case["nu"], g["du"], g["su"], g["DSO"], g["DSD"]
    u = du * (np.arange(nu) + 0.5 - nu / 2.0 + su)
    step, wt = du, np.ones(nu)
    if case["geom"] == "flat":
        q = u * DSO / DSD
        step, wt = du * DSO / DSD, DSO / np.sqrt(DSO ** 2 + q ** 2)
    elif case["geom"] == "arc":
        step, wt = du / DSD, DSO * np.cos(u / DSD)
    # the ramp's taps on a grid zero-padded to a power of two, windowed in frequency
    z = int(2 ** np.ceil(np.log2(2 * nu)))
    k = np.fft.fftfreq(z, d=1.0 / z)
    h = np.zeros(z)
    h[0] = 1.0 / (4.0 * step ** 2)
    h[1::2] = -1.0 / (np.pi ** 2 * step ** 2 * k[1::2] ** 2)
    H, f = step * np.real(np.fft.rfft(h)), np.fft.rfftfreq(z, d=step)
    r = np.minimum(f * 2.0 * step, 1.0)      # frequency over the cutoff 0.5 / step
    H[f > 0.5 / step] = 0.0
    if case["filter"] == "hann":
        H = H * (0.5 + 0.5 * np.cos(np.pi * r))
    elif case["filter"] == "shepp-logan":
        H = H * np.where(r == 0, 1.0, np.sin(np.pi * r / 2) / np.where(r == 0, 1.0, np.pi * r / 2))
    taps = np.fft.irfft(2.0 * H, n=z)[:nu]
    if case["geom"] == "arc":
        q = np.arange(1, nu) * step
        taps[1:] *= (q / np.sin(q)) ** 2
    i = np.arange(nu)
    T = _t(taps[np.abs(i[:, None] - i[None, :])])
    Q = (b.to(F64) * _t(wt)) @ T
    C, S = _trig32(g["ang"])
    x, y = _t(np.arange(case["nx"]) + 0.5 - case["nx"] / 2.0)[:, None], _t(np.arange(case["ny"]) + 0.5 - case["ny"] / 2.0)[None, :]
    out = torch.zeros(case["nx"], case["ny"], dtype=F64, device=DEV)
    c0 = u[0] * step / du
    for a in range(case["views"]):
        c, s = float(C[a]), float(S[a])
        p, den = -s * x + c * y, DSO - (c * x + s * y)
        if case["geom"] == "par":
            pos, w = p, 1.0
        elif case["geom"] == "flat":
            pos, w = DSO / den * p, (DSO / den) ** 2
        else:
            pos, w = torch.atan2(p, den), 1.0 / (den * den + p * p)
        tf = (pos - c0) / step
        fl = torch.floor(tf)
        fr, j = tf - fl, fl.long()
        row = torch.cat([torch.zeros(1, dtype=F64, device=DEV), Q[a], torch.zeros(1, dtype=F64, device=DEV)])
        ok = (j >= -1) & (j <= nu - 1)
        j = (j + 1).clamp(0, nu)
        out += ok * w * ((1 - fr) * row[j] + fr * row[j + 1])
    return out * (np.pi / (2.0 * case["views"]))


def _tv_exact(case, x):
    """Chambolle's dual iteration (J. Math. Imaging Vis. 20, 2004, eq. 9) with
    the documented stopping rule, looked at every ten iterations."""
    g, nd, w = x.to(F64), x.dim(), case["weight"]
    q = [torch.zeros_like(g) for _ in range(nd)]
    tau = 1.0 / (4.0 * nd)

    def div():
        r = torch.zeros_like(g)
        for a in range(nd):
            m = g.shape[a]
            r.narrow(a, 0, m - 1).add_(q[a].narrow(a, 0, m - 1))
            r.narrow(a, 1, m - 1).sub_(q[a].narrow(a, 0, m - 1))
        return r

    for it in range(1, case["most"] + 1):
        v = div() - g
        gr = []
        for a in range(nd):
            m, z = g.shape[a], torch.zeros_like(g)
            z.narrow(a, 0, m - 1).copy_(v.narrow(a, 1, m - 1) - v.narrow(a, 0, m - 1))
            gr.append(z)
        den = 1.0 + tau / w * torch.sqrt(sum(z * z for z in gr))
        most = 0.0
        for a in range(nd):
            new = (q[a] + tau * gr[a]) / den
            if it % 10 == 0:
                most = max(most, float((new - q[a]).abs().max()))
            q[a] = new
        if it % 10 == 0 and most <= 2.0e-4 * w:
            break
    return g - div()


def exact(case, seed):
    op = case["op"]
    if op == "siddon" and _entries(case) > 1.5e9:
        return None          # sorting every ray's planes in float64 takes too long there
    g, data = _inputs(case, seed)
    shape = (case["nx"], case["ny"], case["nz"])
    if op == "tv":
        return _tv_exact(case, data)
    det = (case["views"], case["nu"], case["nv"]) if case["geom"] == "cone" else (case["views"], case["nu"])
    if op == "fbp":
        return _fbp_exact(case, g, data)
    if op == "sf_grad":
        return _sf_grad(case, g, data)
    if op == "siddon_sirt":
        if _entries(case) * (2 + 2 * case["iters"]) > 5e9:
            return None
        return _sirt(_siddon_rows(case, g), data, case["iters"]).reshape(shape)
    if op == "dd_sirt":
        return _sirt(_dd_fan_rows(case, g), data, case["iters"]).reshape(_shape(case))
    if op == "joseph_cone" and _entries(case) > 1.2e10:
        return None
    if op == "joseph_cone":
        y, x = _joseph_cone_pair(case, g, data)
    elif op == "dd_cone":
        y, x = _dd_cone_pair(case, g, data)
    elif op == "sf_cone":
        y, x = _sf_cone_pair(case, g, data)
    else:
        A = {"siddon": _siddon_rows, "sf_fan": _sf_fan_rows, "aw_fan": _aw_fan_rows}[op](case, g)
        y, x = A.pair(data)
    return {"sino": y.reshape(det), "back": x.reshape(shape if op == "siddon" else _shape(case))}
