// Ray-driven projectors for gfx950 (sys_mat/rd.py): Amanatides-Woo voxel
// traversal (path length per voxel) and Joseph interpolation (samples every
// 0.5 length units, bi/trilinear), 2-D parallel, 2-D fan (flat detector)
// and 3-D cone.
//
// Rays (rd.py:472-790): bin centres u = du*(iu - (nu/2 - 0.5) + su) and, for
// the cone, v = dv*(iv - (nu/2 - 0.5) + sv) (the reference centres v with nu);
// parallel rays start at u*(-sin, cos) along (cos, sin); fan/cone rays run
// from the source DSO*(cos, sin, 0) towards the flat detector at
// -(DSD - DSO)*(cos, sin) + u*(-sin, cos) + v*z, unit direction.  [t0, t1] is
// the ray's intersection with the image box (rd.py:51-64, 595-605).
//
// Forward (one thread per ray):
//   AW      sum over voxels of value * intersection length; plane crossings
//           are computed from the plane index (no accumulated t_next += step)
//           and ties step x before y before z (rd.py:111-247); the cone
//           result is scaled by DSD / sqrt(DSD^2 + u^2 + v^2) (rd.py:784-785).
//   Joseph  samples t0 + k/2 <= t1; 2-D clamps the sample into
//           [0, n-2] and interpolates bilinearly (rd.py:250-289); 3-D
//           truncates toward zero and adds only samples whose cell is inside
//           (rd.py:292-353).
// Backward (one thread per voxel, a gather over the rays whose footprint
// can reach it; no atomics): the reference's backprojections (rd.py:151-175,
// 215-247 path-length splat; 356-445 bilinear / trilinear splat with floor
// indices and per-corner bounds), i.e. the transpose of AW's forward (cone:
// without the ray scale), and Joseph's splat.
//
// Rays parallel to an axis (|direction| <= 1e-6) that lie outside the image
// along that axis miss; the reference clamps their entry index onto the
// border row instead (rd.py:66-73), which VIR_COMPAT reproduces: such a ray
// then hits, its index on that axis clamped, and the backprojection also
// visits, for border voxels, the bins whose rays can be axis-parallel.
#include <cmath>

#include "vir_common.h"

namespace vir {

enum RDMode { RD_PAR2 = 0, RD_FAN2 = 1, RD_CONE3 = 2 };
constexpr float kRdEps = 1e-6f;
constexpr float kRdStep = 0.5f;

struct RDGeo {
    int nx, ny, nz, nu, nv, na;
    float d, du, dv, su, sv, DSO, DSD;
    float ucen;   // nu/2 - 0.5 in float32, the bin-centre offset
    float out_scale;
    float bmin[3], bmax[3], c0[3];
    int compat;   // VIR_COMPAT: axis-parallel rays outside the image hit (clamped)
    float inv_du, inv_dv;
    float mar;    // rounding margin of projected bin indices, in bins (rd_u_range)
};

struct RDRay {
    float o[3], h[3];
    float t0, t1;
    float u, v;
    bool hit;
};

__device__ __forceinline__ float rd_ucoord(const RDGeo& G, int iu) {
    return G.du * (((float)iu - G.ucen) + G.su);
}
__device__ __forceinline__ float rd_vcoord(const RDGeo& G, int iv) {
    return G.dv * (((float)iv - G.ucen) + G.sv);
}

template <int MODE>
__device__ __forceinline__ RDRay rd_ray(const RDGeo& G, float c, float s, int iu, int iv) {
    RDRay R;
    const int na = MODE == RD_CONE3 ? 3 : 2;
    R.o[2] = 0.0f;
    R.h[2] = 0.0f;
    R.u = rd_ucoord(G, iu);
    R.v = MODE == RD_CONE3 ? rd_vcoord(G, iv) : 0.0f;
    if (MODE == RD_PAR2) {
        R.o[0] = R.u * -s;
        R.o[1] = R.u * c;
        R.h[0] = c;
        R.h[1] = s;
    } else {
        R.o[0] = G.DSO * c;
        R.o[1] = G.DSO * s;
        const float dx = -(G.DSD - G.DSO) * c + R.u * -s;
        const float dy = -(G.DSD - G.DSO) * s + R.u * c;
        const float vx = dx - R.o[0], vy = dy - R.o[1];
        if (MODE == RD_CONE3) {
            R.o[2] = 0.0f;
            const float vz = R.v;
            const float m = __builtin_sqrtf(vx * vx + vy * vy + vz * vz);
            R.h[0] = vx / m;
            R.h[1] = vy / m;
            R.h[2] = vz / m;
        } else {
            const float m = __builtin_sqrtf(vx * vx + vy * vy);
            R.h[0] = vx / m;
            R.h[1] = vy / m;
        }
    }
    float t0 = -VIR_INF, t1 = VIR_INF;
    bool miss = false;
    for (int a = 0; a < na; ++a) {
        if (fabsf(R.h[a]) > kRdEps) {
            const float ta = (G.bmin[a] - R.o[a]) / R.h[a], tb = (G.bmax[a] - R.o[a]) / R.h[a];
            t0 = fmaxf(t0, fminf(ta, tb));
            t1 = fminf(t1, fmaxf(ta, tb));
        } else if (!(R.o[a] >= G.bmin[a] && R.o[a] < G.bmax[a])) {
            miss = true;
        }
    }
    R.t0 = t0;
    R.t1 = t1;
    R.hit = (!miss || G.compat) && t1 > t0;
    return R;
}

__device__ __forceinline__ int rd_index(const RDGeo& G, int a, float r, int n) {
    r = fminf(fmaxf(r, G.bmin[a] + kRdEps), G.bmax[a] - kRdEps);
    int i = (int)floorf((r - G.bmin[a]) / G.d);
    return min(max(i, 0), n - 1);
}

// ---------------------------------------------------------------- forward

template <int MODE>
__device__ float rd_aw_sum(const RDGeo& G, const RDRay& R, const float* __restrict__ img) {
    const int na = MODE == RD_CONE3 ? 3 : 2;
    const int n[3] = {G.nx, G.ny, MODE == RD_CONE3 ? G.nz : 1};
    int idx[3] = {0, 0, 0}, dir[3] = {0, 0, 0}, nxt[3] = {0, 0, 0};
    float tn[3] = {VIR_INF, VIR_INF, VIR_INF};
    for (int a = 0; a < na; ++a) {
        idx[a] = rd_index(G, a, R.o[a] + R.t0 * R.h[a], n[a]);
        if (fabsf(R.h[a]) > kRdEps) {
            dir[a] = R.h[a] > 0.0f ? 1 : -1;
            nxt[a] = R.h[a] > 0.0f ? idx[a] + 1 : idx[a];
            tn[a] = fmaxf((G.bmin[a] + (float)nxt[a] * G.d - R.o[a]) / R.h[a], R.t0);
        }
    }
    double acc = 0.0;
    float t = R.t0;
    while (t < R.t1) {
        if (idx[0] < 0 || idx[0] >= n[0] || idx[1] < 0 || idx[1] >= n[1] || idx[2] < 0 || idx[2] >= n[2]) break;
        int a;
        if (na == 3) a = (tn[0] <= tn[1] && tn[0] <= tn[2]) ? 0 : (tn[1] <= tn[2] ? 1 : 2);
        else a = tn[0] <= tn[1] ? 0 : 1;
        const float te = fminf(tn[a], R.t1);
        const int64_t vi = na == 3 ? ((int64_t)idx[0] * G.ny + idx[1]) * G.nz + idx[2]
                                   : (int64_t)idx[0] * G.ny + idx[1];
        acc += (double)(img[vi] * (te - t));
        t = te;
        idx[a] += dir[a];
        nxt[a] += dir[a];
        tn[a] = (G.bmin[a] + (float)nxt[a] * G.d - R.o[a]) / R.h[a];
    }
    return (float)acc;
}

template <int MODE>
__device__ float rd_joseph_sum(const RDGeo& G, const RDRay& R, const float* __restrict__ img) {
    double acc = 0.0;
    const float inv_d = 1.0f / G.d;
    for (int k = 0;; ++k) {
        const float t = R.t0 + (float)k * kRdStep;
        if (!(t <= R.t1)) break;
        float fx = (R.o[0] + t * R.h[0] - G.c0[0]) * inv_d;
        float fy = (R.o[1] + t * R.h[1] - G.c0[1]) * inv_d;
        if (MODE != RD_CONE3) {
            fx = fminf(fmaxf(fx, 0.0f), (float)G.nx - 2.0f);
            fy = fminf(fmaxf(fy, 0.0f), (float)G.ny - 2.0f);
            const int ix = (int)fx, iy = (int)fy;
            const float dx = fx - (float)ix, dy = fy - (float)iy;
            const float* p = img + (int64_t)ix * G.ny + iy;
            const float val = p[0] * (1.0f - dx) * (1.0f - dy) + p[G.ny] * dx * (1.0f - dy) +
                              p[1] * (1.0f - dx) * dy + p[G.ny + 1] * dx * dy;
            acc += (double)(val * kRdStep);
        } else {
            const float fz = (R.o[2] + t * R.h[2] - G.c0[2]) * inv_d;
            const int ix = (int)fx, iy = (int)fy, iz = (int)fz;   // truncation, as int() in rd.py
            if (ix >= 0 && ix < G.nx - 1 && iy >= 0 && iy < G.ny - 1 && iz >= 0 && iz < G.nz - 1) {
                const float dx = fx - (float)ix, dy = fy - (float)iy, dz = fz - (float)iz;
                const int64_t sy = G.nz, sx = (int64_t)G.ny * G.nz;
                const float* p = img + ix * sx + iy * sy + iz;
                const float c00 = p[0] + dx * (p[sx] - p[0]);
                const float c10 = p[sy] + dx * (p[sx + sy] - p[sy]);
                const float c01 = p[1] + dx * (p[sx + 1] - p[1]);
                const float c11 = p[sy + 1] + dx * (p[sx + sy + 1] - p[sy + 1]);
                const float c0v = c00 + dy * (c10 - c00);
                const float c1v = c01 + dy * (c11 - c01);
                acc += (double)((c0v + dz * (c1v - c0v)) * kRdStep);
            }
        }
    }
    return (float)acc;
}

template <int MODE, bool JOSEPH>
__global__ __launch_bounds__(256) void k_rd_fp(RDGeo G, const float* __restrict__ cs, const float* __restrict__ sn,
                                              const float* __restrict__ img, float* __restrict__ sino,
                                              int accumulate) {
    const int nv = MODE == RD_CONE3 ? G.nv : 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)G.na * G.nu * nv) return;
    const int iv = (int)(t % nv);
    const int iu = (int)((t / nv) % G.nu);
    const int ia = (int)(t / ((int64_t)nv * G.nu));
    const RDRay R = rd_ray<MODE>(G, cs[ia], sn[ia], iu, iv);
    float val = 0.0f;
    if (R.hit) {
        val = JOSEPH ? rd_joseph_sum<MODE>(G, R, img) : rd_aw_sum<MODE>(G, R, img);
        if (MODE == RD_CONE3 && !JOSEPH)
            val = val * (G.DSD / __builtin_sqrtf(G.DSD * G.DSD + R.u * R.u + R.v * R.v));
    }
    val *= G.out_scale;
    if (accumulate) val += sino[t];
    sino[t] = val;
}

// --------------------------------------------------------------- backward

// Detector coordinates (u, v) of world point (x, y, z) in view (c, s).
template <int MODE>
__device__ __forceinline__ void rd_project(const RDGeo& G, float c, float s, float x, float y, float z, float& u,
                                           float& v) {
    const float p = -s * x + c * y;
    if (MODE == RD_PAR2) {
        u = p;
        v = 0.0f;
        return;
    }
    const float m = G.DSD / (G.DSO - (c * x + s * y));
    u = m * p;
    v = m * z;
}

// Bin index ranges [lo, hi] whose rays can meet the box [x0,x1]x[y0,y1]x[z0,z1].
template <int MODE>
__device__ __forceinline__ void rd_bins(const RDGeo& G, float c, float s, const float* lo, const float* hi, int& u0,
                                        int& u1, int& v0, int& v1) {
    float umin = VIR_INF, umax = -VIR_INF, vmin = VIR_INF, vmax = -VIR_INF;
    const int nc = MODE == RD_CONE3 ? 8 : 4;
    for (int k = 0; k < nc; ++k) {
        float u, v;
        rd_project<MODE>(G, c, s, (k & 1) ? hi[0] : lo[0], (k & 2) ? hi[1] : lo[1], (k & 4) ? hi[2] : lo[2], u, v);
        umin = fminf(umin, u);
        umax = fmaxf(umax, u);
        vmin = fminf(vmin, v);
        vmax = fmaxf(vmax, v);
    }
    const float a0 = umin / G.du + G.ucen - G.su, a1 = umax / G.du + G.ucen - G.su;
    u0 = (int)fmaxf(floorf(a0) - 1.0f, 0.0f);
    u1 = (int)fminf(ceilf(a1) + 1.0f, (float)(G.nu - 1));
    if (!(a1 > -2.0f) || !(a0 < (float)G.nu + 1.0f)) u1 = u0 - 1;
    if (MODE == RD_CONE3) {
        const float b0 = vmin / G.dv + G.ucen - G.sv, b1 = vmax / G.dv + G.ucen - G.sv;
        v0 = (int)fmaxf(floorf(b0) - 1.0f, 0.0f);
        v1 = (int)fminf(ceilf(b1) + 1.0f, (float)(G.nv - 1));
        if (!(b1 > -2.0f) || !(b0 < (float)G.nv + 1.0f)) v1 = v0 - 1;
    } else {
        v0 = 0;
        v1 = 0;
    }
}

// Path length of ray R inside voxel (vx, vy, vz), clipped to [t0, t1].
template <int MODE>
__device__ __forceinline__ float rd_aw_len(const RDGeo& G, const RDRay& R, const int* vi) {
    const int na = MODE == RD_CONE3 ? 3 : 2;
    const int n[3] = {G.nx, G.ny, G.nz};
    float lo = R.t0, hi = R.t1;
    for (int a = 0; a < na; ++a) {
        const float pl = G.bmin[a] + (float)vi[a] * G.d, ph = G.bmin[a] + (float)(vi[a] + 1) * G.d;
        if (fabsf(R.h[a]) > kRdEps) {
            const float ta = (pl - R.o[a]) / R.h[a], tb = (ph - R.o[a]) / R.h[a];
            lo = fmaxf(lo, fminf(ta, tb));
            hi = fminf(hi, fmaxf(ta, tb));
        } else if (rd_index(G, a, R.o[a], n[a]) != vi[a]) {
            return 0.0f;
        }
    }
    return hi > lo ? hi - lo : 0.0f;
}

// Joseph splat weight of ray R into voxel vi (sum over its samples).
template <int MODE>
__device__ __forceinline__ float rd_joseph_w(const RDGeo& G, const RDRay& R, const int* vi) {
    const int na = MODE == RD_CONE3 ? 3 : 2;
    const float inv_d = 1.0f / G.d;
    // samples whose floor cell is vi - 1 or vi on every axis lie in this box
    float lo = R.t0, hi = R.t1;
    for (int a = 0; a < na; ++a) {
        const float pl = G.c0[a] + (float)(vi[a] - 1) * G.d, ph = G.c0[a] + (float)(vi[a] + 1) * G.d;
        if (fabsf(R.h[a]) > kRdEps) {
            const float ta = (pl - R.o[a]) / R.h[a], tb = (ph - R.o[a]) / R.h[a];
            lo = fmaxf(lo, fminf(ta, tb));
            hi = fminf(hi, fmaxf(ta, tb));
        }
    }
    if (!(hi >= lo)) return 0.0f;
    int k0 = (int)fmaxf(floorf((lo - R.t0) / kRdStep) - 1.0f, 0.0f);
    int k1 = (int)floorf((hi - R.t0) / kRdStep) + 1;
    float w = 0.0f;
    for (int k = k0; k <= k1; ++k) {
        const float t = R.t0 + (float)k * kRdStep;
        if (!(t <= R.t1)) break;
        float wk = 1.0f;
        for (int a = 0; a < na; ++a) {
            const float f = (R.o[a] + t * R.h[a] - G.c0[a]) * inv_d;
            const float fl = floorf(f);
            const float dd = f - fl;
            const int i = (int)fl;
            wk *= i == vi[a] ? 1.0f - dd : (i == vi[a] - 1 ? dd : 0.0f);
        }
        w += wk;
    }
    return w * kRdStep;
}

// Bins [b0, b1] of view (c, s) whose rays can run parallel to axis a
// (|h_a| <= kRdEps, rounding included); b1 < b0 when none can.  Parallel
// beam: all bins or none.  Fan/cone: h_a = v_a/|v| with v_x = -DSD c - u s,
// v_y = -DSD s + u c, so |v_a| <= W bounds u to an interval.
template <int MODE>
__device__ void rd_parallel_bins(const RDGeo& G, float c, float s, int a, int& b0, int& b1) {
    b0 = 0;
    b1 = -1;
    if (MODE == RD_PAR2) {
        if (fabsf(a == 0 ? c : s) <= kRdEps) b1 = G.nu - 1;
        return;
    }
    const float k = a == 0 ? -s : c, q = a == 0 ? -G.DSD * c : -G.DSD * s;
    const float umax = fmaxf(fabsf(rd_ucoord(G, 0)), fabsf(rd_ucoord(G, G.nu - 1)));
    const float vmax = MODE == RD_CONE3 ? fmaxf(fabsf(rd_vcoord(G, 0)), fabsf(rd_vcoord(G, G.nv - 1))) : 0.0f;
    const float W = 2e-6f * __builtin_sqrtf(G.DSD * G.DSD + umax * umax + vmax * vmax) + 1e-6f * (G.DSD + umax);
    if (k == 0.0f) {
        if (fabsf(q) <= W) b1 = G.nu - 1;
        return;
    }
    const float ua = (-W - q) / k, ub = (W - q) / k;
    const float fa = fminf(ua, ub) / G.du + G.ucen - G.su, fb = fmaxf(ua, ub) / G.du + G.ucen - G.su;
    b0 = (int)fminf(fmaxf(floorf(fa) - 1.0f, 0.0f), (float)G.nu);
    b1 = (int)fminf(fmaxf(ceilf(fb) + 1.0f, -1.0f), (float)(G.nu - 1));
}

// Adds ray (ia, iu, iv)'s weight on voxel vi times its sinogram value.
template <int MODE, bool JOSEPH>
__device__ __forceinline__ void rd_bp_bin(const RDGeo& G, const float* __restrict__ sino, float c, float s, int ia,
                                          int iu, int iv, const int* vi, double& acc) {
    const int nv = MODE == RD_CONE3 ? G.nv : 1;
    const float y = sino[((int64_t)ia * G.nu + iu) * nv + iv];
    if (y == 0.0f) return;
    const RDRay R = rd_ray<MODE>(G, c, s, iu, iv);
    if (!R.hit) return;
    const float w = JOSEPH ? rd_joseph_w<MODE>(G, R, vi) : rd_aw_len<MODE>(G, R, vi);
    if (w != 0.0f) acc += (double)(y * w);
}

template <int MODE, bool JOSEPH>
__global__ __launch_bounds__(256) void k_rd_bp(RDGeo G, const float* __restrict__ cs, const float* __restrict__ sn,
                                              const float* __restrict__ sino, float* __restrict__ img,
                                              int accumulate) {
    const int nz = MODE == RD_CONE3 ? G.nz : 1, nv = MODE == RD_CONE3 ? G.nv : 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)G.nx * G.ny * nz) return;
    int vi[3];
    vi[2] = (int)(t % nz);
    vi[1] = (int)((t / nz) % G.ny);
    vi[0] = (int)(t / ((int64_t)nz * G.ny));
    // the box whose rays can reach this voxel
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
        if (JOSEPH) {
            lo[a] = G.c0[a] + (float)(vi[a] - 1) * G.d;
            hi[a] = G.c0[a] + (float)(vi[a] + 1) * G.d;
        } else {
            lo[a] = G.bmin[a] + (float)vi[a] * G.d;
            hi[a] = G.bmin[a] + (float)(vi[a] + 1) * G.d;
        }
    }
    if (MODE != RD_CONE3) { lo[2] = 0.0f; hi[2] = 0.0f; }
    // VIR_COMPAT, AW: a ray parallel to axis a outside the image is clamped
    // onto voxel row 0 or n-1 of that axis without passing through it
    const bool edge[2] = {G.compat && !JOSEPH && (vi[0] == 0 || vi[0] == G.nx - 1),
                          G.compat && !JOSEPH && (vi[1] == 0 || vi[1] == G.ny - 1)};
    double acc = 0.0;
    for (int ia = 0; ia < G.na; ++ia) {
        const float c = cs[ia], s = sn[ia];
        int u0, u1, v0, v1;
        rd_bins<MODE>(G, c, s, lo, hi, u0, u1, v0, v1);
        for (int iu = u0; iu <= u1; ++iu)
            for (int iv = v0; iv <= v1; ++iv) rd_bp_bin<MODE, JOSEPH>(G, sino, c, s, ia, iu, iv, vi, acc);
        if (!edge[0] && !edge[1]) continue;
        int e0[2], e1[2];
        for (int a = 0; a < 2; ++a) {
            e0[a] = 0;
            e1[a] = -1;
            if (edge[a]) rd_parallel_bins<MODE>(G, c, s, a, e0[a], e1[a]);
        }
        // every bin of the bands not visited above (nor by the band before)
        for (int a = 0; a < 2; ++a)
            for (int iu = e0[a]; iu <= e1[a]; ++iu) {
                if (a == 1 && iu >= e0[0] && iu <= e1[0]) continue;
                for (int iv = 0; iv < nv; ++iv) {
                    if (iu >= u0 && iu <= u1 && iv >= v0 && iv <= v1) continue;
                    rd_bp_bin<MODE, JOSEPH>(G, sino, c, s, ia, iu, iv, vi, acc);
                }
            }
    }
    float r = (float)acc * G.out_scale;
    if (accumulate) r += img[t];
    img[t] = r;
}

// ------------------------------------------------- backward from ray tables
//
// The per-voxel gather above sets up every ray (a square root and nine
// divisions) again for each voxel and bin it tests, and is bound by that VALU
// work: 74.4 ms for Joseph cone at 128^3, 180 views of 192^2 (6.9 ms here);
// 0.71 ms for path lengths at 129 x 127, 181 views of 223 (0.03 ms here, where
// the views are split over waves as well).  The kernels below
// set each ray up once per block and view, in an LDS table, and leave a voxel
// with the bins its shadow really meets.  Path lengths are the differences of
// the same quotients as in the forward traversal (the pair stays an exact
// transpose).  Joseph's samples are taken in voxel units from the ray's entry
// point: the position there is formed in float64 from the float32 ray and has
// the size of the grid, not of the source distance, so it rounds less than
// o + t h does.  They run over the same k with t0 + k/2 <= t1 in float32 as the
// forward projection's.

// Bins [u0, u1] whose rays can meet the box [x0, x1] x [y0, y1] (the convex
// hull of the projected corners, widened by G.mar for rounding), and the
// least and largest magnification of its corners.  (A view without a finite
// angle: [INT_MAX, INT_MIN].)
template <int MODE>
__device__ __forceinline__ void rd_u_range(const RDGeo& G, float c, float s, float x0, float x1, float y0, float y1,
                                           int& u0, int& u1, float& mmin, float& mmax) {
    float umin = VIR_INF, umax = -VIR_INF;
    mmin = VIR_INF;
    mmax = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float x = (k & 1) ? x1 : x0, y = (k & 2) ? y1 : y0;
        const float p = c * y - s * x;
        float m = 1.0f;
        if (MODE != RD_PAR2) m = G.DSD * __builtin_amdgcn_rcpf(G.DSO - (c * x + s * y));
        umin = fminf(umin, m * p);
        umax = fmaxf(umax, m * p);
        mmin = fminf(mmin, m);
        mmax = fmaxf(mmax, m);
    }
    const float off = G.ucen - G.su;
    u0 = (int)fmaxf(ceilf(umin * G.inv_du + off - G.mar), 0.0f);
    u1 = (int)fminf(floorf(umax * G.inv_du + off + G.mar), (float)(G.nu - 1));
}

// Detector rows [v0, v1] of the heights [z0, z1] at magnifications [mmin, mmax].
__device__ __forceinline__ void rd_v_range(const RDGeo& G, float z0, float z1, float mmin, float mmax, int& v0,
                                           int& v1) {
    const float off = G.ucen - G.sv;
    const float lo = z0 * (z0 < 0.0f ? mmax : mmin), hi = z1 * (z1 < 0.0f ? mmin : mmax);
    v0 = (int)fmaxf(ceilf(lo * G.inv_dv + off - G.mar), 0.0f);
    v1 = (int)fminf(floorf(hi * G.inv_dv + off + G.mar), (float)(G.nv - 1));
}

// A ray of an LDS table.  Joseph: position at t0 (p) and step per sample (h)
// in voxels, the reciprocals of the step (r) and the last sample's index (t1).
// Path lengths: origin, direction and its reciprocal in world units and
// [t0, t1], so that plane crossings come out as the forward traversal's
// quotients.  t1 < t0: dead.
template <int NA>
struct RDTab {
    float p[NA], h[NA], r[NA], t0, t1, y;
};

template <int MODE, bool JOSEPH, int NA>
__device__ __forceinline__ RDTab<NA> rd_tab(const RDGeo& G, float c, float s, int iu, int iv, float y) {
    const int n[3] = {G.nx, G.ny, G.nz};
    RDTab<NA> T;
    T.y = y;
    T.t0 = 0.0f;
    T.t1 = -1.0f;
    const RDRay R = rd_ray<MODE>(G, c, s, iu, iv);
    const bool live = R.hit && y != 0.0f;
    const double inv_d = 1.0 / (double)G.d;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        if (JOSEPH) {
            T.p[a] = (float)(((double)R.o[a] + (double)R.t0 * (double)R.h[a] - (double)G.c0[a]) * inv_d);
            T.h[a] = (float)((double)(kRdStep * R.h[a]) * inv_d);
        } else {
            T.p[a] = R.o[a];
            T.h[a] = R.h[a];
            if (!(fabsf(R.h[a]) > kRdEps)) {  // parallel to the axis: in one voxel row, from its centre
                T.p[a] = G.bmin[a] + ((float)rd_index(G, a, R.o[a], n[a]) + 0.5f) * G.d;
                T.h[a] = 1e-30f;
            }
        }
        // finite reciprocals: a ray that does not move along an axis gets
        // interval ends far beyond [t0, t1], both of one sign outside
        T.r[a] = fminf(fmaxf(1.0f / T.h[a], -1e30f), 1e30f);
    }
    if (!live) return T;
    if (JOSEPH) {
        int k = (int)((R.t1 - R.t0) * (1.0f / kRdStep));
        // (bounded: far sources, where t0 + 1/2 rounds to t0, end it too)
        for (int i = 0; i < 65536 && R.t0 + (float)(k + 1) * kRdStep <= R.t1; ++i) ++k;
        while (k > 0 && !(R.t0 + (float)k * kRdStep <= R.t1)) --k;
        T.t1 = (float)k;
    } else {
        T.t0 = R.t0;
        T.t1 = R.t1;
    }
    return T;
}

// a / b from the correctly rounded reciprocal r of b (Markstein's correction)
__device__ __forceinline__ float rd_quot(float a, float b, float r) {
    const float q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), r, q);
}

// The voxel a lane works on: index coordinates (Joseph) or its lower and
// upper planes (path lengths).
template <bool JOSEPH>
__device__ __forceinline__ void rd_voxel(const RDGeo& G, int a, int i, float& f0, float& f1) {
    f0 = JOSEPH ? (float)i : G.bmin[a] + (float)i * G.d;
    f1 = JOSEPH ? 0.0f : G.bmin[a] + (float)(i + 1) * G.d;
}

// Weight of a table ray on that voxel: the summed hat-function products of
// its samples (Joseph; samples outside the voxel's 2-voxel box weigh zero, so
// the sample range only has to cover it), or its path length.
template <bool JOSEPH, int NA>
__device__ __forceinline__ float rd_tab_w(const RDTab<NA>& T, const float* f0, const float* f1) {
    float x[NA], lo = T.t0, hi = T.t1;
    if (!JOSEPH) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const float p = rd_quot(f0[a] - T.p[a], T.h[a], T.r[a]), q = rd_quot(f1[a] - T.p[a], T.h[a], T.r[a]);
            lo = fmaxf(lo, fminf(p, q));
            hi = fminf(hi, fmaxf(p, q));
        }
        return hi > lo ? hi - lo : 0.0f;
    }
    float pl = -VIR_INF, ph = VIR_INF;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        x[a] = T.p[a] - f0[a];
        const float p = (-1.0f - x[a]) * T.r[a], q = (1.0f - x[a]) * T.r[a];
        pl = fmaxf(pl, fminf(p, q));
        ph = fminf(ph, fmaxf(p, q));
    }
    lo = fmaxf(lo, ceilf(pl - 0.02f));
    hi = fminf(hi, floorf(ph + 0.02f));
    float w = 0.0f;
    for (float k = lo; k <= hi; k += 1.0f) {
        float wk = 1.0f;
#pragma unroll
        for (int a = 0; a < NA; ++a)
            wk *= fmaxf(1.0f - fabsf(__builtin_fmaf(k, T.h[a], x[a])), 0.0f);
        w += wk;
    }
    return w * kRdStep;
}

// Cone beam: a block of eight waves takes 8 x NC columns of 64 voxels, NC
// columns a wave (lane = voxel of the column), one view at a time.
constexpr int kRdWaves = 8;
constexpr int kRdCap = 832;  // rays of one table: 39 KiB, four blocks a CU

template <bool JOSEPH, int NC>
__global__ __launch_bounds__(64 * kRdWaves) void k_rd_bp_cone_tab(RDGeo G, const float* __restrict__ cs,
                                                                 const float* __restrict__ sn,
                                                                 const float* __restrict__ sino,
                                                                 float* __restrict__ img, int accumulate, int nby,
                                                                 int nbz) {
    // columns x = bx .. bx + 3, y = by .. by + 2 NC - 1
    constexpr int BX = 4, BY = 2 * NC, NCOL = BX * BY;
    __shared__ float4 ta[kRdCap], tb[kRdCap], tc[kRdCap];
    __shared__ int cu0[NCOL], cu1[NCOL];
    __shared__ float cm0[NCOL], cm1[NCOL];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int blk = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int bz = (blk % nbz) * 64;
    blk /= nbz;
    const int by = (blk % nby) * BY, bx = (blk / nby) * BX;
    const int iz = bz + lane;
    // the box of voxel index range [i, j] along axis a: voxels (path length)
    // or one voxel around the centres (Joseph)
    auto box_lo = [&](int a, int i) { return JOSEPH ? G.c0[a] + (float)(i - 1) * G.d : G.bmin[a] + (float)i * G.d; };
    auto box_hi = [&](int a, int j) { return JOSEPH ? G.c0[a] + (float)(j + 1) * G.d : G.bmin[a] + (float)(j + 1) * G.d; };
    const int ex = min(bx + BX, G.nx) - 1, ey = min(by + BY, G.ny) - 1, ez = min(bz + 64, G.nz) - 1;
    const float X0 = box_lo(0, bx), X1 = box_hi(0, ex), Y0 = box_lo(1, by), Y1 = box_hi(1, ey);
    const float Z0 = box_lo(2, bz), Z1 = box_hi(2, ez);
    const float z0 = box_lo(2, iz), z1 = box_hi(2, iz);
    double acc[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) acc[q] = 0.0;
    for (int ia = 0; ia < G.na; ++ia) {
        const float c = cs[ia], s = sn[ia];
        int U0, U1, V0, V1;
        float m0, m1;
        rd_u_range<RD_CONE3>(G, c, s, X0, X1, Y0, Y1, U0, U1, m0, m1);
        rd_v_range(G, Z0, Z1, m0, m1, V0, V1);
        if (U1 < U0 || V1 < V0) continue;  // the same in every thread
        const int cv = min(V1 - V0 + 1, kRdCap), cu = min(U1 - U0 + 1, kRdCap / cv);
        const float* plane = sino + (int64_t)ia * G.nu * G.nv;
        for (int ub = U0; ub <= U1; ub += cu)
            for (int vb = V0; vb <= V1; vb += cv) {
                const int ue = min(ub + cu - 1, U1), ve = min(vb + cv - 1, V1);
                __syncthreads();  // the table's last readers are done
                for (int e = tid; e < (ue - ub + 1) * cv; e += 64 * kRdWaves) {
                    const int iu = ub + e / cv, iv = vb + e % cv;
                    const bool in = iv <= ve;
                    const RDTab<3> T = rd_tab<RD_CONE3, JOSEPH, 3>(G, c, s, iu, iv, in ? plane[(int64_t)iu * G.nv + iv] : 0.0f);
                    ta[e] = make_float4(T.p[0], T.p[1], T.p[2], T.y);
                    tb[e] = make_float4(T.r[0], T.r[1], T.r[2], T.t1);
                    tc[e] = make_float4(T.h[0], T.h[1], T.h[2], T.t0);
                }
                if (tid < NCOL) {
                    const int ix = bx + tid % BX, iy = by + tid / BX;
                    rd_u_range<RD_CONE3>(G, c, s, box_lo(0, ix), box_hi(0, ix), box_lo(1, iy), box_hi(1, iy), cu0[tid],
                                         cu1[tid], cm0[tid], cm1[tid]);
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    const int col = wave + kRdWaves * q;  // x = col % BX, y = col / BX
                    float f0[3], f1[3];
                    rd_voxel<JOSEPH>(G, 0, bx + col % BX, f0[0], f1[0]);
                    rd_voxel<JOSEPH>(G, 1, by + col / BX, f0[1], f1[1]);
                    rd_voxel<JOSEPH>(G, 2, iz, f0[2], f1[2]);
                    int v0, v1;
                    rd_v_range(G, z0, z1, cm0[col], cm1[col], v0, v1);
                    v0 = max(v0, vb);
                    v1 = min(v1, ve);
                    if (iz >= G.nz) v1 = -1;
                    const int u1 = min(cu1[col], ue);
                    for (int iu = max(cu0[col], ub); iu <= u1; ++iu)
                        for (int iv = v0; iv <= v1; ++iv) {
                            const int e = (iu - ub) * cv + iv - vb;
                            const float4 a = ta[e], b = tb[e], h = tc[e];
                            const RDTab<3> T = {{a.x, a.y, a.z}, {h.x, h.y, h.z}, {b.x, b.y, b.z}, h.w, b.w, a.w};
                            const float w = rd_tab_w<JOSEPH, 3>(T, f0, f1);
                            if (w != 0.0f) acc[q] += (double)(T.y * w);
                        }
                }
            }
    }
    if (iz >= G.nz) return;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const int col = wave + kRdWaves * q;
        const int ix = bx + col % BX, iy = by + col / BX;
        if (ix >= G.nx || iy >= G.ny) continue;
        const int64_t o = ((int64_t)ix * G.ny + iy) * G.nz + iz;
        float r = (float)acc[q] * G.out_scale;
        if (accumulate) r += img[o];
        img[o] = r;
    }
}

// Parallel and fan beam: a block takes a tile of 16 x 8 pixels, two a lane;
// its NW waves share the views (wave w takes the view pairs w, w + NW, ...)
// and keep a table each, so the view loop has no barrier; the waves' float64
// sums are added in wave order.  A table holds 32 rays of two views; a tile
// that meets more is done in several rounds.
constexpr int kRd2X = 16, kRd2Y = 8;

template <int MODE, bool JOSEPH, int NW>
__global__ __launch_bounds__(64 * NW) void k_rd_bp_2d_tab(RDGeo G, const float* __restrict__ cs,
                                                          const float* __restrict__ sn,
                                                          const float* __restrict__ sino, float* __restrict__ img,
                                                          int accumulate, int nby) {
    __shared__ float4 tab[NW][64][2];
    __shared__ float tab_y[NW][64];
    __shared__ double part[NW][kRd2X * kRd2Y];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = (blockIdx.x / nby) * kRd2X, by = (blockIdx.x % nby) * kRd2Y;
    auto box_lo = [&](int a, int i) { return JOSEPH ? G.c0[a] + (float)(i - 1) * G.d : G.bmin[a] + (float)i * G.d; };
    auto box_hi = [&](int a, int j) { return JOSEPH ? G.c0[a] + (float)(j + 1) * G.d : G.bmin[a] + (float)(j + 1) * G.d; };
    const float X0 = box_lo(0, bx), X1 = box_hi(0, min(bx + kRd2X, G.nx) - 1);
    const float Y0 = box_lo(1, by), Y1 = box_hi(1, min(by + kRd2Y, G.ny) - 1);
    // this lane's pixels: (bx + lane / 8, by + lane % 8) and eight rows on
    const int ix = bx + (lane >> 3), iy = by + (lane & 7);
    const int slot = lane >> 5, j = lane & 31;
    float4(*t)[2] = tab[wave];
    float* ty = tab_y[wave];
    double acc[2] = {0.0, 0.0};
    for (int a0 = 2 * wave; a0 < G.na; a0 += 2 * NW) {
        const int ia = min(a0 + slot, G.na - 1);
        int U0, U1;
        float m0, m1;
        rd_u_range<MODE>(G, cs[ia], sn[ia], X0, X1, Y0, Y1, U0, U1, m0, m1);
        U0 = min(U0, G.nu);   // lengths and indexes below don't overflow
        U1 = max(U1, -1);
        if (a0 + slot >= G.na) U1 = U0 - 1;
        // the two views' ranges, the same in every lane
        const int A0 = __builtin_amdgcn_readlane(U0, 0), A1 = __builtin_amdgcn_readlane(U1, 0);
        const int B0 = __builtin_amdgcn_readlane(U0, 32), B1 = __builtin_amdgcn_readlane(U1, 32);
        const int rounds = (max(max(A1 - A0, B1 - B0), -1) + 32) / 32;
        for (int rd = 0; rd < rounds; ++rd) {
            const int iu = U0 + 32 * rd + j;
            if (iu <= U1) {
                const RDTab<2> T = rd_tab<MODE, JOSEPH, 2>(G, cs[ia], sn[ia], iu, 0, sino[(int64_t)ia * G.nu + iu]);
                t[lane][0] = make_float4(T.p[0], T.p[1], T.t0, T.t1);
                t[lane][1] = make_float4(T.r[0], T.r[1], T.h[0], T.h[1]);
                ty[lane] = T.y;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a wave's LDS accesses are in order
#pragma unroll
            for (int sl = 0; sl < 2; ++sl) {
                const int base = (sl ? B0 : A0) + 32 * rd, end = min(base + 31, sl ? B1 : A1);
                if (end < base) continue;
                const float c = cs[a0 + sl], s = sn[a0 + sl];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int px = ix + 8 * q;
                    int u0, u1;
                    rd_u_range<MODE>(G, c, s, box_lo(0, px), box_hi(0, px), box_lo(1, iy), box_hi(1, iy), u0, u1, m0, m1);
                    u0 = max(u0, base);
                    u1 = min(u1, end);
                    float f0[2], f1[2];
                    rd_voxel<JOSEPH>(G, 0, px, f0[0], f1[0]);
                    rd_voxel<JOSEPH>(G, 1, iy, f0[1], f1[1]);
                    for (int u = u0; u <= u1; ++u) {
                        const int e = 32 * sl + u - base;
                        const float4 a = t[e][0], b = t[e][1];
                        const RDTab<2> T = {{a.x, a.y}, {b.z, b.w}, {b.x, b.y}, a.z, a.w, ty[e]};
                        const float w = rd_tab_w<JOSEPH, 2>(T, f0, f1);
                        if (w != 0.0f) acc[q] += (double)(T.y * w);
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    part[wave][lane] = acc[0];
    part[wave][64 + lane] = acc[1];
    __syncthreads();
    for (int e = tid; e < kRd2X * kRd2Y; e += 64 * NW) {
        const int px = bx + (e >> 3), py = by + (e & 7);
        if (px >= G.nx || py >= G.ny) continue;
        double sum = part[0][e];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += part[w][e];
        const int64_t o = (int64_t)px * G.ny + py;
        float r = (float)sum * G.out_scale;
        if (accumulate) r += img[o];
        img[o] = r;
    }
}

static int rd_setup(const vir_rd_geom* g, RDGeo& G) {
    if (!g) return fail_arg("geometry is NULL");
    if (g->mode < 0 || g->mode > 2) return fail_arg("mode must be 0 (par), 1 (fan) or 2 (cone)");
    const bool is3 = g->mode == RD_CONE3;
    G.nx = g->nx; G.ny = g->ny; G.nz = is3 ? g->nz : 1;
    G.nu = g->nu; G.nv = is3 ? g->nv : 1; G.na = g->na;
    G.d = g->d_pix; G.du = g->du; G.dv = is3 ? g->dv : 1.0f; G.su = g->su; G.sv = is3 ? g->sv : 0.0f;
    G.DSO = g->DSO; G.DSD = g->DSD;
    G.compat = 0;
    if (G.nx < 2 || G.ny < 2 || G.nz < 1 || (is3 && G.nz < 2) || G.nu < 1 || G.nv < 1 || G.na < 0)
        return fail_arg("bad sizes (image axes need >= 2 voxels)");
    if (!(G.d > 0.0f) || !(G.du > 0.0f) || !(G.dv > 0.0f)) return fail_arg("spacings must be > 0");
    G.ucen = (float)(0.5 * (double)G.nu - 0.5);
    const int n[3] = {G.nx, G.ny, G.nz};
    for (int a = 0; a < 3; ++a) {
        G.bmin[a] = -G.d * (float)n[a] / 2.0f;
        G.bmax[a] = G.d * (float)n[a] / 2.0f;
        G.c0[a] = -G.d * ((float)n[a] / 2.0f - 0.5f);
    }
    G.inv_du = 1.0f / G.du;
    G.inv_dv = 1.0f / G.dv;
    if (g->mode != RD_PAR2) {
        if (!(G.DSO > 0.0f) || !(G.DSD > G.DSO)) return fail_arg("need 0 < DSO < DSD");
        const double hx = 0.5 * G.nx * (double)G.d, hy = 0.5 * G.ny * (double)G.d;
        if (!(std::sqrt(hx * hx + hy * hy) + 2.0 * G.d < G.DSO)) return fail_arg("grid reaches the source");
    }
    // bin indices are sums of terms as large as the detector, its offset and
    // the grid's shadow (in bins): a few float32 roundings of those
    const double hz = 0.5 * G.nz * (double)G.d, hr = std::sqrt(0.25 * ((double)G.nx * G.nx + (double)G.ny * G.ny)) * G.d;
    const double mag = g->mode == RD_PAR2 ? 1.0 : (double)G.DSD / (G.DSO - hr - G.d);
    const double terms = (double)G.nu + G.nv + std::fabs((double)G.su) + std::fabs((double)G.sv) +
                         mag * (hr / G.du + (is3 ? hz / G.dv : 0.0));
    G.mar = (float)(0.02 + 2e-6 * terms);
    return VIR_OK;
}

// False where the table kernels do not apply, and for cone-beam volumes so thin
// that theirs, whose 64 lanes run along z, is slower than one thread per voxel:
// two slabs, or three with interpolation, in bricks enough to fill the chip.
// Table | per voxel, us, 60 views, slabs: Joseph 128^2 (512 bricks) 2: equal; 150^2
// (722) 2: 1206 | 1140; 180^2 (1035) 2: 1704 | 1142, 3: 2251 | 1964; 220^2 3: 3123 |
// 2484, 4: 3108 | 3453; path lengths 180^2 2: 629 | 617, 256^2 2: 983 | 787, 3: 990 |
// 1426.
static bool rd_tab_pays(const RDGeo& G, int mode, bool jo) {
    // samples are counted in float32 there: exactly, and so that the count ends,
    // below 2^24, a ray of 8.4 million units (grids in very small units)
    const double nz = mode == RD_CONE3 ? G.nz : 0.0;
    if (jo && std::sqrt((double)G.nx * G.nx + (double)G.ny * G.ny + nz * nz) * G.d > 8e6) return false;
    // (a launch can't have more threads)
    const int64_t blocks = mode == RD_CONE3 ? (int64_t)((G.nx + 3) / 4) * ((G.ny + 7) / 8) * ((G.nz + 63) / 64)
                                            : (int64_t)((G.nx + kRd2X - 1) / kRd2X) * ((G.ny + kRd2Y - 1) / kRd2Y);
    if (blocks * (mode == RD_CONE3 ? 64 * kRdWaves : 256) > kLaunchThreads) return false;
    if (mode != RD_CONE3 || G.nz > (jo ? 3 : 2)) return true;
    return (int64_t)((G.nx + 3) / 4) * ((G.ny + 7) / 8) < (jo && G.nz == 2 ? 650 : 1000);
}

// The table kernels' launch.  Cone: four columns a wave (a 4 x 8 x 64 brick,
// its rays set up once per 2048 voxels) where that gives the chip two blocks
// a CU, else one column a wave.  2-D: sixteen waves share a tile's views
// while the tiles alone would leave CUs idle, else four.
static int rd_bp_tab(const RDGeo& G, int mode, bool jo, const float* cosv, const float* sinv, const float* sino,
                     float* img, int acc, hipStream_t st) {
    if (mode == RD_CONE3) {
        const int nbx = (G.nx + 3) / 4, nbz = (G.nz + 63) / 64;
        const bool wide = (int64_t)nbx * ((G.ny + 7) / 8) * nbz >= 512;
        const int nby = wide ? (G.ny + 7) / 8 : (G.ny + 1) / 2;
        const dim3 grd((unsigned)((int64_t)nbx * nby * nbz)), blk(64 * kRdWaves);
        if (jo && wide)
            hipLaunchKernelGGL((k_rd_bp_cone_tab<true, 4>), grd, blk, 0, st, G, cosv, sinv, sino, img, acc, nby, nbz);
        else if (jo)
            hipLaunchKernelGGL((k_rd_bp_cone_tab<true, 1>), grd, blk, 0, st, G, cosv, sinv, sino, img, acc, nby, nbz);
        else if (wide)
            hipLaunchKernelGGL((k_rd_bp_cone_tab<false, 4>), grd, blk, 0, st, G, cosv, sinv, sino, img, acc, nby, nbz);
        else
            hipLaunchKernelGGL((k_rd_bp_cone_tab<false, 1>), grd, blk, 0, st, G, cosv, sinv, sino, img, acc, nby, nbz);
        return check_hip(hipGetLastError(), "vir_rd_bp launch");
    }
    const int nbx = (G.nx + kRd2X - 1) / kRd2X, nby = (G.ny + kRd2Y - 1) / kRd2Y;
    const int64_t tiles = (int64_t)nbx * nby;
    const bool many = tiles >= 1024;
    const dim3 grd((unsigned)tiles);
#define VIR_RD_BP2(M, J)                                                                                            \
    do {                                                                                                            \
        if (many)                                                                                                   \
            hipLaunchKernelGGL((k_rd_bp_2d_tab<M, J, 4>), grd, dim3(256), 0, st, G, cosv, sinv, sino, img, acc, nby);  \
        else                                                                                                        \
            hipLaunchKernelGGL((k_rd_bp_2d_tab<M, J, 16>), grd, dim3(1024), 0, st, G, cosv, sinv, sino, img, acc, nby); \
    } while (0)
    if (mode == RD_PAR2) {
        if (jo) VIR_RD_BP2(RD_PAR2, true);
        else VIR_RD_BP2(RD_PAR2, false);
    } else {
        if (jo) VIR_RD_BP2(RD_FAN2, true);
        else VIR_RD_BP2(RD_FAN2, false);
    }
#undef VIR_RD_BP2
    return check_hip(hipGetLastError(), "vir_rd_bp launch");
}

}  // namespace vir

using namespace vir;

extern "C" {

int vir_rd_fp(const vir_rd_geom* geom, const float* cosv, const float* sinv, const float* img, float* sino,
              float out_scale, uint32_t flags, void* stream) {
    RDGeo G;
    int rc = rd_setup(geom, G);
    if (rc) return rc;
    if (G.na == 0) return VIR_OK;
    if (!cosv || !sinv || !img || !sino) return fail_arg("NULL pointer argument");
    G.out_scale = out_scale;
    G.compat = (flags & VIR_COMPAT) ? 1 : 0;
    const int64_t n = (int64_t)G.na * G.nu * G.nv;
    dim3 grd((unsigned)((n + 255) / 256));
    hipStream_t st = as_stream(stream);
    const int acc = (flags & VIR_ACCUMULATE) ? 1 : 0;
    const bool jo = geom->joseph != 0;
#define VIR_RD_FP(M)                                                                                        \
    do {                                                                                                      \
        if (jo) hipLaunchKernelGGL((k_rd_fp<M, true>), grd, dim3(256), 0, st, G, cosv, sinv, img, sino, acc);  \
        else hipLaunchKernelGGL((k_rd_fp<M, false>), grd, dim3(256), 0, st, G, cosv, sinv, img, sino, acc);   \
    } while (0)
    if (geom->mode == RD_PAR2) VIR_RD_FP(RD_PAR2);
    else if (geom->mode == RD_FAN2) VIR_RD_FP(RD_FAN2);
    else VIR_RD_FP(RD_CONE3);
#undef VIR_RD_FP
    return check_hip(hipGetLastError(), "vir_rd_fp launch");
}

int vir_rd_bp(const vir_rd_geom* geom, const float* cosv, const float* sinv, const float* sino, float* img,
              float out_scale, uint32_t flags, void* stream) {
    RDGeo G;
    int rc = rd_setup(geom, G);
    if (rc) return rc;
    if ((G.na > 0 && (!cosv || !sinv || !sino)) || !img) return fail_arg("NULL pointer argument");
    G.out_scale = out_scale;
    G.compat = (flags & VIR_COMPAT) ? 1 : 0;
    const int acc = (flags & VIR_ACCUMULATE) ? 1 : 0;
    const bool jo = geom->joseph != 0;
    hipStream_t st = as_stream(stream);
    // VIR_COMPAT's clamped rays reach voxels they do not pass through: only
    // the per-voxel gather visits those
    if (!G.compat && !(flags & VIR_PER_OUTPUT) && rd_tab_pays(G, geom->mode, jo))
        return rd_bp_tab(G, geom->mode, jo, cosv, sinv, sino, img, acc, st);
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    dim3 grd((unsigned)((n + 255) / 256));
#define VIR_RD_BP(M)                                                                                        \
    do {                                                                                                      \
        if (jo) hipLaunchKernelGGL((k_rd_bp<M, true>), grd, dim3(256), 0, st, G, cosv, sinv, sino, img, acc);  \
        else hipLaunchKernelGGL((k_rd_bp<M, false>), grd, dim3(256), 0, st, G, cosv, sinv, sino, img, acc);   \
    } while (0)
    if (geom->mode == RD_PAR2) VIR_RD_BP(RD_PAR2);
    else if (geom->mode == RD_FAN2) VIR_RD_BP(RD_FAN2);
    else VIR_RD_BP(RD_CONE3);
#undef VIR_RD_BP
    return check_hip(hipGetLastError(), "vir_rd_bp launch");
}

}  // extern "C"
