// Pixel-driven separable-footprint projectors for gfx950 (sys_mat/pd.py):
// 2-D parallel and fan, 3-D cone, and a batched 3-D parallel variant whose
// detector rows run along z.
//
// Footprint model: each pixel's four corners are projected onto the detector
// and the pixel deposits over [min, max] of them with amplitude
//   parallel : 1/(|sin| + |cos|)                           (pd.py:181)
//   fan      : 1/(|cos(a+g)| + |sin(a+g)|), g = atan(u_c/DSD) (pd.py:292-298)
//   cone     : 1/(|sin| + |cos|), u from the four parallel-projected
//              corners times the centre's fan magnification, v from the
//              slab bounds times magnification/cos(g)   (pd.py:423-451)
// weight per bin = overlap/du (* overlap_v/dv); the forward output is
// scaled by d_pix (pd.py:234, 350, 485).
//
// Forward: a (batch, view, bin[, row]) gathers the pixels whose footprints meet
// the bin (centre projection inverted along the driving axis, widened by the
// largest footprint half-width).  Backward: a (batch, pixel[, slab]) visits the
// bins its footprint meets.  No atomics.  One thread per output (VIR_PER_OUTPUT,
// and where nothing else applies) every weight comes from the same functions in
// both directions, an exact transpose.  Most calls take tiles: flat_tile.h (2-D),
// cone_tile.h, and for parallel 3-D the matrix kernels below, whose footprints are
// the same but whose overlaps are formed in their own units and order, so that
// the pair is a transpose to the float32 rounding of the weights.
//
// VIR_COMPAT (fan forward only): the reference skips a zero pixel without
// advancing its o boundary (pd.py:321-325), so the next nonzero pixel's
// amplitude takes its lower y boundary from just after the previous nonzero
// pixel of the column (the first boundary if none); footprints are unchanged.
#include <cmath>
#include <type_traits>

#include "cone_tile.h"
#include "flat_tile.h"
#include "vir_common.h"

namespace vir {

enum SFMode { SF_PAR2 = 0, SF_FAN2 = 1, SF_CONE3 = 2, SF_PAR3 = 3 };

struct SFGeo {
    int nx, ny, nz, nu, nv, na, nb;
    float d, du, dv, su, sv, DSO, DSD;
    float out_scale;
    float wmax;  // largest footprint half-width along u (detector units)
    int unit_amp;  // parallel modes: amplitude 1 (VIR_SF_UNIT_AMPLITUDE)
    int compat;    // fan forward: stale o boundary after zero pixels (VIR_COMPAT)
};

__device__ __forceinline__ float sf_bnd(int n, float d, int k) { return d * ((float)k - 0.5f * (float)n); }
__device__ __forceinline__ float sf_det(int n, float du, float su, int j) {
    return du * (((float)j - 0.5f * (float)n) + su);
}

struct SFFoot {
    float u0, u1;   // footprint along u
    float amp;      // amplitude
    float cm;       // v magnification (cone) or 1
};

// Per-view constants.
struct SFView {
    float c, s;
    float ca, sa;  // cosine and sine of the float32 angle (fan amplitude)
    float amp;     // 1/(|sin| + |cos|)
    float h;       // half the projected width of a pixel in parallel beam
};

__device__ __forceinline__ SFView sf_view(const SFGeo& G, float c, float s, float ang) {
    SFView V;
    V.c = c;
    V.s = s;
    V.ca = cosf(ang);
    V.sa = sinf(ang);
    const float w = fabsf(s) + fabsf(c);
    V.amp = G.unit_amp ? 1.0f : 1.0f / w;
    V.h = 0.5f * G.d * w;
    return V;
}

// Fan amplitude 1/(|cos(a+g)| + |sin(a+g)|) of pixel (ix, iy), g the angle
// of the ray through its centre, whose o coordinate takes the pixel's lower
// y boundary at boundary ky (ky = iy: the pixel's own).  With t = tan g it is
// sqrt(1 + t^2) / (|cos a - t sin a| + |sin a + t cos a|): no trigonometry per
// pixel, and no rounding of a + g.
__device__ __forceinline__ float sf_fan_amp(const SFGeo& G, const SFView& V, int ix, int iy, int ky) {
    const float c = V.c, s = V.s;
    const float xl = sf_bnd(G.nx, G.d, ix), xr = sf_bnd(G.nx, G.d, ix + 1);
    const float yl = sf_bnd(G.ny, G.d, iy), yr = sf_bnd(G.ny, G.d, iy + 1);
    const float pxc = (-s * xl + -s * xr) * 0.5f, oxc = (c * xl + c * xr) * 0.5f;
    const float pyc = (c * yl + c * yr) * 0.5f, oyc = (s * sf_bnd(G.ny, G.d, ky) + s * yr) * 0.5f;
    const float t = (pxc + pyc) / (G.DSO - (oxc + oyc));
    return __builtin_sqrtf(1.0f + t * t) / (fabsf(V.ca - t * V.sa) + fabsf(V.sa + t * V.ca));
}

// Footprint of pixel (ix, iy) in view V.  In parallel beam the four
// projected corners -s*x + c*y span exactly [p_c - h, p_c + h] around the
// centre's projection p_c, h = d(|sin| + |cos|)/2.
template <int MODE>
__device__ __forceinline__ SFFoot sf_foot(const SFGeo& G, const SFView& V, int ix, int iy) {
    const float c = V.c, s = V.s;
    SFFoot f;
    f.cm = 1.0f;
    f.amp = V.amp;
    if (MODE == SF_PAR2 || MODE == SF_PAR3) {
        const float xc = G.d * (((float)ix + 0.5f) - 0.5f * (float)G.nx);
        const float yc = G.d * (((float)iy + 0.5f) - 0.5f * (float)G.ny);
        const float pc = -s * xc + c * yc;
        f.u0 = pc - V.h;
        f.u1 = pc + V.h;
        return f;
    }
    const float xl = sf_bnd(G.nx, G.d, ix), xr = sf_bnd(G.nx, G.d, ix + 1);
    const float yl = sf_bnd(G.ny, G.d, iy), yr = sf_bnd(G.ny, G.d, iy + 1);
    const float pxl = -s * xl, pxr = -s * xr, pyl = c * yl, pyr = c * yr;
    const float oxl = c * xl, oxr = c * xr, oyl = s * yl, oyr = s * yr;
    if (MODE == SF_FAN2) {
        float p0 = G.DSD * (pxl + pyl) / (G.DSO - (oxl + oyl));
        float p1 = G.DSD * (pxr + pyl) / (G.DSO - (oxr + oyl));
        float p2 = G.DSD * (pxl + pyr) / (G.DSO - (oxl + oyr));
        float p3 = G.DSD * (pxr + pyr) / (G.DSO - (oxr + oyr));
        f.u0 = fminf(fminf(p0, p1), fminf(p2, p3));
        f.u1 = fmaxf(fmaxf(p0, p1), fmaxf(p2, p3));
        f.amp = sf_fan_amp(G, V, ix, iy, iy);
        return f;
    }
    // cone
    const float pxc = (pxl + pxr) * 0.5f, oxc = (oxl + oxr) * 0.5f;
    const float pyc = (pyl + pyr) * 0.5f, oyc = (oyl + oyr) * 0.5f;
    const float den_c = G.DSO - (oxc + oyc);
    const float fm = G.DSD / den_c;
    float u0 = fm * (pxl + pyl), u1 = fm * (pxr + pyl), u2 = fm * (pxl + pyr), u3 = fm * (pxr + pyr);
    f.u0 = fminf(fminf(u0, u1), fminf(u2, u3));
    f.u1 = fmaxf(fmaxf(u0, u1), fmaxf(u2, u3));
    // over the cosine of the fan angle atan(t): sqrt(1 + t^2) as 1 + t^2 / (1 +
    // sqrt(1 + t^2)), whose small term's rounding hardly counts
    const float t = (pxc + pyc) / den_c, t2 = t * t;
    f.cm = __builtin_fmaf(fm, t2 * __builtin_amdgcn_rcpf(1.0f + __builtin_sqrtf(1.0f + t2)), fm);
    return f;
}

// Rows (FP: slabs) a slab (row) of the parallel 3-D geometry meets, with
// their weights overlap/dv: independent of the pixel and the view, so
// computed once per thread.  Up to kSlabs entries -- enough for rows no
// taller than a voxel, rounding included; more (taller rows) fall back to
// the general loop.
constexpr int kSlabs = 5;
struct SlabWeights {
    int first, count;
    float w[kSlabs];
};

__device__ __forceinline__ float ovl(float a0, float a1, float b0, float b1) {
    return fminf(a1, b1) - fmaxf(a0, b0);
}

// Slabs that detector row iv of the parallel 3-D geometry meets, with their
// weights overlap/dv (zero-padded to kSlabs).  Returns false when the row
// meets more than kSlabs slabs (rows taller than a voxel).
__device__ __forceinline__ bool par3_row_slabs(const SFGeo& G, int iv, SlabWeights& SW) {
    const float vl = sf_det(G.nv, G.dv, G.sv, iv), vr = sf_det(G.nv, G.dv, G.sv, iv + 1);
    const float inv_d = 1.0f / G.d, inv_dv = 1.0f / G.dv;
    float z0f = fminf(vl, vr) * inv_d + 0.5f * (float)G.nz;
    float z1f = fmaxf(vl, vr) * inv_d + 0.5f * (float)G.nz;
    int z0 = (int)fmaxf(floorf(z0f) - 1.0f, 0.0f);
    int z1 = (int)fminf(floorf(z1f) + 1.0f, (float)(G.nz - 1));
    SW.first = z0;
    SW.count = z1 - z0 + 1;
    if (z1 - z0 + 1 > kSlabs) {
#pragma unroll
        for (int k = 0; k < kSlabs; ++k) SW.w[k] = 0.0f;
        return false;
    }
#pragma unroll
    for (int k = 0; k < kSlabs; ++k) {
        const int z = z0 + k;
        float ov = z <= z1 ? ovl(sf_bnd(G.nz, G.d, z), sf_bnd(G.nz, G.d, z + 1), vl, vr) : 0.0f;
        SW.w[k] = ov > 0.0f ? ov * inv_dv : 0.0f;
    }
    return true;
}

// Detector rows that slab iz of the parallel 3-D geometry meets, with their
// weights overlap/dv (zero-padded to kSlabs).  Returns false when the slab
// meets more than kSlabs rows (rows much shorter than a voxel).
__device__ __forceinline__ bool par3_slab_rows(const SFGeo& G, int iz, SlabWeights& SW) {
    const float zl = sf_bnd(G.nz, G.d, iz), zr = sf_bnd(G.nz, G.d, iz + 1);
    const float v0 = sf_det(G.nv, G.dv, G.sv, 0), inv_dv = 1.0f / G.dv;
    const float lo = fminf(zl, zr), hi = fmaxf(zl, zr);
    int m0 = (int)fmaxf(floorf((lo - v0) * inv_dv) - 1.0f, 0.0f);
    int m1 = (int)fminf(floorf((hi - v0) * inv_dv) + 1.0f, (float)(G.nv - 1));
    SW.first = m0;
    SW.count = m1 - m0 + 1;
    if (m1 - m0 + 1 > kSlabs) {
#pragma unroll
        for (int k = 0; k < kSlabs; ++k) SW.w[k] = 0.0f;
        return false;
    }
#pragma unroll
    for (int k = 0; k < kSlabs; ++k) {
        const int m = m0 + k;
        float ov = m <= m1 ? ovl(zl, zr, sf_det(G.nv, G.dv, G.sv, m), sf_det(G.nv, G.dv, G.sv, m + 1)) : 0.0f;
        SW.w[k] = ov > 0.0f ? ov * inv_dv : 0.0f;
    }
    return true;
}

// centre projection along the driving axis, inverted: the drive coordinate
// whose pixel centre projects to u on orthogonal line coordinate oc
template <int MODE>
__device__ __forceinline__ float sf_invert(const SFGeo& G, bool xd, float c, float s, float u, float oc) {
    // p = pd*drive + po*orth, o = od*drive + oo*orth (o toward the source)
    float pd = xd ? -s : c, po = xd ? c : -s;
    float od = xd ? c : s, oo = xd ? s : c;
    if (MODE == SF_PAR2 || MODE == SF_PAR3) return (u - po * oc) / pd;
    float t = u / G.DSD;
    return (t * (G.DSO - oo * oc) - po * oc) / (pd + t * od);
}

// One view of the 2-D geometries as flat_tile.h's model.  The forward tile
// adds the terms of k_sf_fp in float64 as that kernel does, grouped by wave.
template <int MODE>
struct SFFlat {
    static constexpr int kFixed = 4;
    static constexpr bool kShared = false, kCentre = true, kCorners = MODE == SF_FAN2;
    struct Trig {
        SFView V;
        __device__ Trig(float c, float s, float ang) {
            V.c = c;
            V.s = s;
            V.ca = MODE == SF_FAN2 ? cosf(ang) : 0.0f;
            V.sa = MODE == SF_FAN2 ? sinf(ang) : 0.0f;
        }
        __device__ Trig lane(int l) const {
            Trig t = *this;
            t.V.c = ft_lane(V.c, l);
            t.V.s = ft_lane(V.s, l);
            t.V.ca = ft_lane(V.ca, l);
            t.V.sa = ft_lane(V.sa, l);
            return t;
        }
    };
    const SFGeo& G;
    SFView V;
    bool xd;
    int nd, no;
    __device__ SFFlat(const SFGeo& g, const Trig& t) : G(g), V(t.V) {
        const float w = fabsf(V.s) + fabsf(V.c);
        V.amp = G.unit_amp ? 1.0f : 1.0f / w;
        V.h = 0.5f * G.d * w;
        xd = fabsf(V.s) >= fabsf(V.c);
        nd = xd ? G.nx : G.ny;
        no = xd ? G.ny : G.nx;
    }
    __device__ float centre(int io) const { return (sf_bnd(no, G.d, io) + sf_bnd(no, G.d, io + 1)) * 0.5f; }
    __device__ float lin(float u, float& A, float& B) const {
        const float pd = xd ? -V.s : V.c, po = xd ? V.c : -V.s;
        const float od = xd ? V.c : V.s, oo = xd ? V.s : V.c;
        const float t = MODE == SF_PAR2 ? u : u / G.DSD, den = MODE == SF_PAR2 ? pd : pd + t * od, r = 1.0f / den;
        A = MODE == SF_PAR2 ? t * r : t * G.DSO * r;
        B = MODE == SF_PAR2 ? po * r : (t * oo + po) * r;
        return den;
    }
    __device__ float margin() const { return G.wmax; }
    __device__ float line_factor(float) const { return 1.0f / G.du; }
    __device__ float pixel(int k, int io, float& u0, float& u1) const {
        const SFFoot f = sf_foot<MODE>(G, V, xd ? k : io, xd ? io : k);
        u0 = f.u0;
        u1 = f.u1;
        return f.amp;
    }
    __device__ float amp(int k, int io) const { return sf_fan_amp(G, V, xd ? k : io, xd ? io : k, xd ? io : k); }
    __device__ float grid(int k, int io) const { return xd ? corner(k, io) : corner(io, k); }
    __device__ float corner(int ix, int iy) const {
        const float x = sf_bnd(G.nx, G.d, ix), y = sf_bnd(G.ny, G.d, iy);
        return G.DSD * (-V.s * x + V.c * y) / (G.DSO - (V.c * x + V.s * y));
    }
    // pixel (ix + i, iy + j) at 2 i + j; a fan block has nine corners
    __device__ void quad(int ix, int iy, float* lo, float* hi, float* f) const {
        float p[3][3];
        if (MODE == SF_FAN2) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) p[i][j] = corner(ix + i, iy + j);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = q >> 1, j = q & 1;
            if (MODE == SF_PAR2) {
                const SFFoot t = sf_foot<SF_PAR2>(G, V, ix + i, iy + j);
                lo[q] = t.u0;
                hi[q] = t.u1;
                f[q] = t.amp;
                continue;
            }
            lo[q] = fminf(fminf(p[i][j], p[i + 1][j]), fminf(p[i][j + 1], p[i + 1][j + 1]));
            hi[q] = fmaxf(fmaxf(p[i][j], p[i + 1][j]), fmaxf(p[i][j + 1], p[i + 1][j + 1]));
            f[q] = sf_fan_amp(G, V, ix + i, iy + j, iy + j);
        }
    }
    __host__ __device__ static float bp_unit(const SFGeo& g) { return 1.0f / g.du; }
};

// One view of the cone geometry as cone_tile.h's model: weights and ranges of
// the one-thread-per-output kernels below.
struct SFCone {
    static constexpr bool kLineMag = false;
    const SFGeo& G;
    SFView V;
    bool xd;
    int nd, no;
    __device__ SFCone(const SFGeo& g, float c, float s, float ang) : G(g), V(sf_view(g, c, s, ang)) {
        xd = fabsf(s) >= fabsf(c);
        nd = xd ? G.nx : G.ny;
        no = xd ? G.ny : G.nx;
    }
    __device__ bool range(float ul, float ur, int io, int& k0, int& k1) const {
        const float oc = (sf_bnd(no, G.d, io) + sf_bnd(no, G.d, io + 1)) * 0.5f, inv_d = 1.0f / G.d;
        const float x0 = sf_invert<SF_CONE3>(G, xd, V.c, V.s, ul - G.wmax, oc);
        const float x1 = sf_invert<SF_CONE3>(G, xd, V.c, V.s, ur + G.wmax, oc);
        const float k0f = fminf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        const float k1f = fmaxf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        if (!(k0f < (float)nd + 1.0f) || !(k1f > -2.0f)) return false;
        k0 = (int)fmaxf(floorf(k0f) - 1.0f, 0.0f);
        k1 = (int)fminf(floorf(k1f) + 2.0f, (float)(nd - 1));
        return true;
    }
    __device__ SFFoot at(int k, int io) const { return sf_foot<SF_CONE3>(G, V, xd ? k : io, xd ? io : k); }
    __device__ void foot(int k, int io, float& lo, float& hi) const {
        const SFFoot f = at(k, io);
        lo = f.u0;
        hi = f.u1;
    }
    __device__ float weight(int k, int io, float ul, float ur) const {
        const SFFoot f = at(k, io);
        return ((fminf(f.u1, ur) - fmaxf(f.u0, ul)) * (1.0f / G.du)) * f.amp;
    }
    __device__ float zmag(int k, int io) const { return at(k, io).cm; }
    __host__ __device__ static float fp_unit(const SFGeo& g) { return 1.0f / g.dv; }
    __host__ __device__ static float bp_unit(const SFGeo&) { return 1.0f; }
};

template <int MODE>
__global__ __launch_bounds__(256) void k_sf_fp(SFGeo G, const float* __restrict__ ang,
                                              const float* __restrict__ cs, const float* __restrict__ sn,
                                              const float* __restrict__ img, float* __restrict__ sino,
                                              int accumulate) {
    const bool is3 = MODE == SF_CONE3 || MODE == SF_PAR3;
    const int nv = is3 ? G.nv : 1;
    const int64_t per_b = (int64_t)G.na * G.nu * nv;
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= per_b * G.nb) return;
    const int b = (int)(t / per_b);
    int64_t r = t % per_b;
    const int iv = (int)(r % nv);
    const int iu = (int)((r / nv) % G.nu);
    const int ia = (int)(r / ((int64_t)nv * G.nu));
    const SFView V = sf_view(G, cs[ia], sn[ia], ang[ia]);
    const float c = V.c, s = V.s;
    const bool xd = fabsf(s) >= fabsf(c);
    const int nd = xd ? G.nx : G.ny, no = xd ? G.ny : G.nx;
    const float ul = sf_det(G.nu, G.du, G.su, iu), ur = sf_det(G.nu, G.du, G.su, iu + 1);
    const float vl = sf_det(nv, G.dv, G.sv, iv), vr = sf_det(nv, G.dv, G.sv, iv + 1);
    const float inv_d = 1.0f / G.d, inv_du = 1.0f / G.du, inv_dv = 1.0f / G.dv;
    const int nz = is3 ? G.nz : 1;
    const float* vol = img + (int64_t)b * G.nx * G.ny * nz;
    // parallel 3-D: the slabs of this detector row and their weights
    SlabWeights SW;
    SW.first = 0;
    SW.count = 0;
    bool slab_general = false;
    if (MODE == SF_PAR3) slab_general = !par3_row_slabs(G, iv, SW);
    double acc = 0.0;
    const auto line = [&](int io) {
        const float oc = (sf_bnd(no, G.d, io) + sf_bnd(no, G.d, io + 1)) * 0.5f;
        float x0 = sf_invert<MODE>(G, xd, c, s, ul - G.wmax, oc);
        float x1 = sf_invert<MODE>(G, xd, c, s, ur + G.wmax, oc);
        float k0f = fminf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        float k1f = fmaxf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        if (!(k0f < (float)nd + 1.0f) || !(k1f > -2.0f)) return;
        int k0 = (int)fmaxf(floorf(k0f) - 1.0f, 0.0f);
        int k1 = (int)fminf(floorf(k1f) + 2.0f, (float)(nd - 1));
        for (int k = k0; k <= k1; ++k) {
            const int ix = xd ? k : io, iy = xd ? io : k;
            const SFFoot f = sf_foot<MODE>(G, V, ix, iy);
            const float ou = ovl(f.u0, f.u1, ul, ur);
            if (!(ou > 0.0f)) continue;
            float wu = (ou * inv_du) * f.amp;
            const float* col = vol + ((int64_t)ix * G.ny + iy) * nz;
            if (MODE == SF_FAN2 && G.compat && col[0] != 0.0f) {
                // the last nonzero pixel before iy in column ix
                int j = iy - 1;
                while (j >= 0 && vol[(int64_t)ix * G.ny + j] == 0.0f) --j;
                if (j + 1 != iy) wu = (ou * inv_du) * sf_fan_amp(G, V, ix, iy, j + 1);
            }
            if (!is3) {
                acc += (double)(col[0] * wu);
            } else if (MODE == SF_PAR3 && !slab_general) {
                float sv_ = 0.0f;
#pragma unroll
                for (int q = 0; q < kSlabs; ++q)
                    if (SW.w[q] > 0.0f) sv_ += col[SW.first + q] * SW.w[q];
                acc = __builtin_fma((double)wu, (double)sv_, acc);
            } else {
                // slabs whose magnified z interval meets [vl, vr]
                float z0f = fminf(vl, vr) / f.cm * inv_d + 0.5f * (float)G.nz;
                float z1f = fmaxf(vl, vr) / f.cm * inv_d + 0.5f * (float)G.nz;
                int z0 = (int)fmaxf(floorf(z0f) - 1.0f, 0.0f);
                int z1 = (int)fminf(floorf(z1f) + 1.0f, (float)(G.nz - 1));
                for (int z = z0; z <= z1; ++z) {
                    float ov = ovl(f.cm * sf_bnd(G.nz, G.d, z), f.cm * sf_bnd(G.nz, G.d, z + 1), vl, vr);
                    if (ov > 0.0f) acc += (double)(col[z] * (wu * (ov * inv_dv)));
                }
            }
        }
    };
    if (is3) {
        for (int io = 0; io < no; ++io) line(io);
    } else {
        // in the tile's chains of lines: the same bits
        double sum = 0.0;
        for (int w = 0; w < 4; ++w) {
            double part = 0.0;
            for (int c = w; c < kFtLines; c += 4) {
                acc = 0.0;
                for (int io = c; io < no; io += kFtLines) line(io);
                part += acc;
            }
            sum += part;
        }
        acc = sum;
    }
    float res = (float)acc * G.out_scale;
    if (accumulate) res += sino[t];
    sino[t] = res;
}

// ------------------------------------------ tiled parallel 3-D forward
//
// A block computes 16 bins x 64 detector rows of four neighbouring views of one
// batch item, one view per wave.  For every orthogonal line the rows' slab sums
//   P[k][m] = sum over the row's slabs q of w_q(m) * vox[k][first(m) + q]
// of the pixels whose footprints can meet the tile in any of the views are
// brought into LDS (P depends on the line and the pixel only, so the views
// share it), and each wave adds its view's footprint weights times P as
// float64 matrix products (v_mfma_f64_4x4x4_4b_f64: exact products of the
// float32 factors, float64 sums).  Its four blocks take four groups of four
// bins, each with the pixel window its group meets: 4 du plus a footprint, six
// to eight pixels, so two K-steps of four pixels for pixels as wide as bins,
// and a third of the products count.  A lane evaluates the weight its operand
// slot needs and reads the same pixel's rows: no lists, no broadcasts.
//
// Each of NG wave groups takes every NG-th chunk of a line's pixels; their sums
// are added at the end in group order.
//
// Rows that meet exactly one slab with weight 1 (UNIT) need no slab sums: the
// voxel rows go straight from memory into the LDS operand, the next line's
// while a line is multiplied, with one barrier a line.  Otherwise each wave
// replaces its share of the staged rows by their slab sums in place.
//
// The matrix and vector operations of the waves take turns: 16 products a K-step
// (294 cycles of about 500, with the 16 conversions, one weight and the reads).
// Staging more lines ahead changed nothing; more than five waves a SIMD were not
// to be had (16 float64 sums a lane).  8 x 256 x 256 x 64, 180 views of 384 x 64:
// 8.2 -> 3.0 ms against a form that listed each bin's pixels with cross-lane
// prefix sums and accumulated row by row; 1 x 256 x 256 x 64, 64 views, 2.79 -> 0.50.
constexpr int kTUB = 16;  // detector bins per tile and view
constexpr int kVG = 4;    // views per workgroup (one per wave)
constexpr int kTV = 64;   // detector rows per tile
constexpr int kMK = 40;   // pixels of one line staged at once
constexpr int kMP = 68;   // LDS row pitch: 16-byte reads of four windows of rows meet different banks
constexpr int kZW = 66;   // slabs a tile's 64 rows can meet (rows no taller than a voxel: 65)

// One bin and row by the gather.
__device__ double sf_fp_par3_one(const SFGeo& G, const SFView& V, const float* __restrict__ vol, int iu, int iv) {
    const bool xd = fabsf(V.s) >= fabsf(V.c);
    const int nd = xd ? G.nx : G.ny, no = xd ? G.ny : G.nx;
    const float ul = sf_det(G.nu, G.du, G.su, iu), ur = sf_det(G.nu, G.du, G.su, iu + 1);
    const float inv_d = 1.0f / G.d, inv_du = 1.0f / G.du;
    SlabWeights SW;
    par3_row_slabs(G, iv, SW);
    double acc = 0.0;
    for (int io = 0; io < no; ++io) {
        const float oc = (sf_bnd(no, G.d, io) + sf_bnd(no, G.d, io + 1)) * 0.5f;
        const float x0 = sf_invert<SF_PAR3>(G, xd, V.c, V.s, ul - G.wmax, oc);
        const float x1 = sf_invert<SF_PAR3>(G, xd, V.c, V.s, ur + G.wmax, oc);
        const float k0f = fminf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        const float k1f = fmaxf(x0, x1) * inv_d + 0.5f * (float)nd - 0.5f;
        if (!(k0f < (float)nd + 1.0f) || !(k1f > -2.0f)) continue;
        const int k0 = (int)fmaxf(floorf(k0f) - 1.0f, 0.0f), k1 = (int)fminf(floorf(k1f) + 2.0f, (float)(nd - 1));
        for (int k = k0; k <= k1; ++k) {
            const int ix = xd ? k : io, iy = xd ? io : k;
            const SFFoot f = sf_foot<SF_PAR3>(G, V, ix, iy);
            const float ou = ovl(f.u0, f.u1, ul, ur);
            if (!(ou > 0.0f)) continue;
            const float* col = vol + ((int64_t)ix * G.ny + iy) * G.nz;
            float sv = 0.0f;
#pragma unroll
            for (int q = 0; q < kSlabs; ++q)
                if (SW.w[q] > 0.0f) sv += col[SW.first + q] * SW.w[q];
            acc = __builtin_fma((double)((ou * inv_du) * f.amp), (double)sv, acc);
        }
    }
    return acc;
}

template <bool UNIT, int NG>
__global__ __launch_bounds__(64 * kVG * NG) __attribute__((amdgpu_waves_per_eu(4))) void k_sf_fp_par3_mfma(SFGeo G, const float* __restrict__ cs,
                                                             const float* __restrict__ sn,
                                                             const float* __restrict__ img, float* __restrict__ sino,
                                                             int accumulate, int nut, int nmt, int nvg, int shift) {
    // two objects, so that reads of one need not wait for loads into the other
    __shared__ __attribute__((aligned(16))) float R0[NG * kMK * kMP], R1[NG * kMK * kMP];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % kVG;
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / kVG;
    // operand slots: group (matrix block) mid; weights: bin lo, pixel hi; rows:
    // row quad lo, pixel hi; sums: bin hi, row quad lo
    const int lo = lane & 3, mid = (lane >> 2) & 3, hi = lane >> 4;
    int blk = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int m_lo = (blk % nmt) * kTV;
    blk /= nmt;
    const int u_lo = (blk % nut) * kTUB;
    blk /= nut;
    const int a0 = (blk % nvg) * kVG, nva = min(kVG, G.na - a0);
    const int b = blk / nvg;
    const int ia = a0 + min(wave, nva - 1);
    const bool vwave = wave < nva;
    const SFView V = sf_view(G, cs[ia], sn[ia], 0.0f);
    const bool xd = fabsf(V.s) >= fabsf(V.c);
    const float inv_d = 1.0f / G.d, inv_du = 1.0f / G.du;
    const float* vol = img + (int64_t)b * G.nx * G.ny * G.nz;

    // staging lanes: row m_lo + lane.  UNIT: its slab; else the slabs of
    // non-zero weight in slab order, and the tile's slab range zb, span
    const int m = m_lo + lane;
    bool zin = false;
    int zb = 0, span = 64, nzs = 0, zo[kSlabs];
    float swt[kSlabs];
    if (UNIT) {
        zb = m_lo - shift;
        zin = m < G.nv && zb + lane >= 0 && zb + lane < G.nz;
    } else {
        SlabWeights SW;
        par3_row_slabs(G, min(m, G.nv - 1), SW);
        int sz[kSlabs];
#pragma unroll
        for (int q = 0; q < kSlabs; ++q) {
            sz[q] = 0;
            swt[q] = 0.0f;
        }
#pragma unroll
        for (int q = 0; q < kSlabs; ++q) {
            if (SW.w[q] > 0.0f) {
#pragma unroll
                for (int r = 0; r < kSlabs; ++r) {  // slot nzs, without dynamic register indexing
                    if (r == nzs) {
                        sz[r] = SW.first + q;
                        swt[r] = SW.w[q];
                    }
                }
                ++nzs;
            }
        }
        if (m >= G.nv) nzs = 0;
        int zlo = 0x7fffffff, zhi = -1;
#pragma unroll
        for (int q = 0; q < kSlabs; ++q)
            if (q < nzs) {
                zlo = min(zlo, sz[q]);
                zhi = max(zhi, sz[q]);
            }
#pragma unroll
        for (int t = 32; t >= 1; t >>= 1) {
            zlo = min(zlo, __shfl_xor(zlo, t));
            zhi = max(zhi, __shfl_xor(zhi, t));
        }
        zb = __builtin_amdgcn_readfirstlane(zhi >= 0 ? zlo : 0);
        span = min(__builtin_amdgcn_readfirstlane(zhi >= 0 ? zhi - zlo + 1 : 0), kZW);
#pragma unroll
        for (int q = 0; q < kSlabs; ++q) zo[q] = min(max(sz[q] - zb, 0), kZW - 1);
    }

    // this lane's weight: bin u_lo + 4 mid + lo; its group's pixel window
    // starts at the first centre that projects past the group's left edge less
    // a half footprint (x = A - oc B in pixels, widened by its rounding)
    const int iu = u_lo + 4 * mid + lo;
    const float ul = sf_det(G.nu, G.du, G.su, iu), ur = sf_det(G.nu, G.du, G.su, iu + 1);
    const float pd = xd ? -V.s : V.c, po = xd ? V.c : -V.s;
    const int nd = xd ? G.nx : G.ny;
    const float eps = 2e-3f + 2e-6f * (float)(G.nx + G.ny);
    const float rp = inv_d / pd, gB = po * rp, gc = 0.5f * (float)nd - 0.5f - eps;
    const float ge0 = (sf_det(G.nu, G.du, G.su, u_lo + 4 * mid) - V.h) * rp;
    const float ge1 = (sf_det(G.nu, G.du, G.su, u_lo + 4 * mid + 4) + V.h) * rp;
    const float gA = fminf(ge0, ge1) + gc;
    const int nks = __builtin_amdgcn_readfirstlane(((int)floorf(fabsf(ge1 - ge0) + 2.0f * eps) + 4) >> 2);

    // the tile's edges, and the views' bands x = at0 - oc lin .. at1 - oc lin
    const float ut0 = sf_det(G.nu, G.du, G.su, u_lo), ut1 = sf_det(G.nu, G.du, G.su, min(u_lo + kTUB, G.nu));
    bool gxd[kVG], mixed = false;
    float glin[kVG], gat0[kVG], gat1[kVG];
#pragma unroll
    for (int w = 0; w < kVG; ++w) {
        const int aw = a0 + min(w, nva - 1);
        const SFView W = sf_view(G, cs[aw], sn[aw], 0.0f);
        gxd[w] = fabsf(W.s) >= fabsf(W.c);
        const float ipd = inv_d / (gxd[w] ? -W.s : W.c);
        glin[w] = (gxd[w] ? W.c : -W.s) * ipd;
        const float e0 = (ut0 - W.h) * ipd, e1 = (ut1 + W.h) * ipd;
        gat0[w] = fminf(e0, e1) - eps;
        gat1[w] = fmaxf(e0, e1) + eps;
        mixed |= w < nva && gxd[w] != gxd[0];
    }

    double acc[16];  // bin u_lo + 4 mid + hi, rows 16 c + 4 lo + e at 4 c + e
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0;

    // views whose driving axis is that of the first view, then the others
    for (int pass = 0; pass < (mixed ? 2 : 1); ++pass) {
        const bool pxd = pass == 0 ? gxd[0] : !gxd[0];
        // (a view without a finite angle meets nothing)
        const bool active = vwave && xd == pxd && fabsf(V.c) + fabsf(V.s) < VIR_INF;
        const int pnd = pxd ? G.nx : G.ny, pno = pxd ? G.ny : G.nx;
        const int64_t kstride = (int64_t)(pxd ? G.ny : 1) * G.nz, lstride = (int64_t)(pxd ? 1 : G.ny) * G.nz;
        for (int lb = 0; lb < pno; lb += 64) {
            // lane = line lb + lane: the union of the pass's views' pixel bands
            const int iol = lb + lane;
            const float ocl = (sf_bnd(pno, G.d, iol) + sf_bnd(pno, G.d, iol + 1)) * 0.5f;
            int k0l = pnd, k1l = -1;
#pragma unroll
            for (int w = 0; w < kVG; ++w) {
                if (w >= nva || gxd[w] != pxd) continue;
                const float c0 = 0.5f * (float)pnd - 0.5f;
                k0l = min(k0l, (int)fmaxf(ceilf(__builtin_fmaf(-ocl, glin[w], gat0[w]) + c0), 0.0f));
                k1l = max(k1l, (int)fminf(floorf(__builtin_fmaf(-ocl, glin[w], gat1[w]) + c0), (float)(pnd - 1)));
            }
            if (iol >= pno) k1l = -1;
            // this group's chunk (line cl, pixels ck .., nk of them; of every
            // NG the group's own): all groups walk the same list
            int l = -1, kc = 0, ke = -1, cl = 0, ck = 0, nk = 0;
            const auto stage = [&](float* dst) {
                bool any = false;
                nk = 0;
#pragma unroll
                for (int s = 0; s < NG; ++s) {
                    kc += kMK;
                    while (kc > ke && l < 64) {
                        if (++l >= 64 || lb + l >= pno) {
                            l = 64;
                            break;
                        }
                        kc = __builtin_amdgcn_readlane(k0l, l);
                        ke = __builtin_amdgcn_readlane(k1l, l);
                    }
                    any |= l < 64;
                    if (s == grp && l < 64) {
                        cl = l;
                        ck = kc;
                        nk = min(kMK, ke - kc + 1);
                    }
                }
                const float* p = vol + (int64_t)(lb + cl) * lstride + (int64_t)ck * kstride + zb + lane;
                for (int kk = wave; kk < nk; kk += kVG) {
                    float* row = dst + (grp * kMK + kk) * kMP;
                    if (UNIT ? zin : lane < span)
                        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + kk * kstride),
                                                         (__attribute__((address_space(3))) void*)row, 4, 0, 0);
                    if (!UNIT && lane < span - 64)
                        __builtin_amdgcn_global_load_lds(
                            (const __attribute__((address_space(1))) void*)(p + kk * kstride + 64),
                            (__attribute__((address_space(3))) void*)(row + 64), 4, 0, 0);
                }
                return any;
            };
            __syncthreads();  // the last chunk's readers are done
            bool more = stage(R0);
            const auto step = [&](float* Rp, float* Rn) {
                const int dl = cl, dk = ck, dn = nk;
                Rp += grp * kMK * kMP;
                __syncthreads();  // these chunks have landed; the other buffer is no longer read
                more = stage(Rn);
                if (!UNIT) {
                    // slab sums of this wave's rows, in place: each row is read
                    // and rewritten by one wave, reads before writes
                    for (int kk = wave; kk < dn; kk += kVG) {
                        float sv = 0.0f;
#pragma unroll
                        for (int q = 0; q < kSlabs; ++q)
                            if (q < nzs) sv += Rp[kk * kMP + zo[q]] * swt[q];
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        Rp[kk * kMP + lane] = sv;
                    }
                    __syncthreads();
                }
                if (!active || dn == 0) return;
                const float oc = ct_lane(ocl, dl);
                const float xl = G.d * (((float)(lb + dl) + 0.5f) - 0.5f * (float)pno);
                const int win = (int)ceilf(__builtin_fmaf(-oc, gB, gA)) + hi;
                for (int kk = 0; kk < nks; ++kk) {
                    const int k = win + 4 * kk, kr = k - dk;
                    const float xk = G.d * (((float)k + 0.5f) - 0.5f * (float)nd);
                    const float pc = pd * xk + po * xl;
                    const float ou = ovl(pc - V.h, pc + V.h, ul, ur);
                    const bool in = ou > 0.0f && (unsigned)kr < (unsigned)dn;
                    if (!__any(in)) continue;  // another view's pixels, or another chunk's
                    const double w = in ? (double)((ou * inv_du) * V.amp) : 0.0;
                    const float4* row = (const float4*)(Rp + min(max(kr, 0), dn - 1) * kMP + 4 * lo);
                    float4 x[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) x[c] = row[4 * c];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        acc[4 * c] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, (double)x[c].x, acc[4 * c], 0, 0, 0);
                        acc[4 * c + 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, (double)x[c].y, acc[4 * c + 1], 0, 0, 0);
                        acc[4 * c + 2] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, (double)x[c].z, acc[4 * c + 2], 0, 0, 0);
                        acc[4 * c + 3] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, (double)x[c].w, acc[4 * c + 3], 0, 0, 0);
                    }
                }
            };
            while (more) {
                step(R0, R1);
                if (more) step(R1, R0);
            }
        }
    }
    // the groups' sums, in group order
    static_assert(NG == 1 || kVG * 64 * 8 * 2 <= NG * kMK * kMP, "eight sums a lane fit a buffer");
#pragma unroll
    for (int g = 1; g < NG; ++g) {
        double *S0 = (double*)R0 + wave * 512 + lane, *S1 = (double*)R1 + wave * 512 + lane;
        __syncthreads();
        if (grp == g) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                S0[64 * i] = acc[i];
                S1[64 * i] = acc[8 + i];
            }
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                acc[i] += S0[64 * i];
                acc[8 + i] += S1[64 * i];
            }
        }
    }
    if (grp != 0) return;
    const int ob = u_lo + 4 * mid + hi;
    if (!vwave || ob >= G.nu) return;
    float* out = sino + (((int64_t)b * G.na + ia) * G.nu + ob) * G.nv;
    const auto put = [&](int mr, double v) {
        const float res = (float)v * G.out_scale;
        out[mr] = accumulate ? out[mr] + res : res;
    };
    unsigned odd = 0;  // sums with zero weights times infinities: by the gather
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int mr = m_lo + 16 * (i >> 2) + 4 * lo + (i & 3);
        if (mr >= G.nv) continue;
        if (UNIT && (mr - shift < 0 || mr - shift >= G.nz)) put(mr, 0.0);  // a row without a slab
        else if (fabs(acc[i]) < (double)VIR_INF) put(mr, acc[i]);
        else odd |= 1u << i;
    }
    while (odd) {
        const int i = __ffs((int)odd) - 1;
        odd &= odd - 1;
        const int mr = m_lo + 16 * (i >> 2) + 4 * lo + (i & 3);
        put(mr, sf_fp_par3_one(G, V, vol, ob, mr));
    }
}

// ------------------------------------------ parallel 3-D backward by columns
//
// One wave per (batch item, pixel, 64 slabs): lane z accumulates voxel z of
// the column over all views.  The footprint of the pixel -- bins with
// positive overlap and their weights -- is computed for 64 views at once
// (lane = view) and broadcast with readlane in the view loop, which then only
// reads the sinogram rows each slab meets (consecutive lanes, consecutive
// rows) and accumulates.  Weights, bin and view order and arithmetic are
// those of k_sf_bp, so both give the same bits.  The kernel waits on memory:
// the rows of a view's first kJPre bins are loaded together, and 64 VGPRs
// keep eight waves per SIMD.
constexpr int kJMax = 8;  // bins a pixel footprint meets (checked on the host)
constexpr int kJPre = 2;  // bins whose sinogram rows are loaded together

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_sf_bp_par3_col(SFGeo G, const float* __restrict__ ang,
                                                       const float* __restrict__ cs,
                                                       const float* __restrict__ sn,
                                                       const float* __restrict__ sino, float* __restrict__ img,
                                                       int accumulate, int nzt) {
    const int lane = threadIdx.x & 63;
    const int64_t wid = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wid >= (int64_t)G.nb * G.nx * G.ny * nzt) return;  // whole wave
    const int zt = (int)(wid % nzt);
    int64_t r = wid / nzt;
    const int iy = (int)(r % G.ny);
    r /= G.ny;
    const int ix = (int)(r % G.nx);
    const int b = (int)(r / G.nx);
    const int iz = zt * 64 + lane;
    const bool zin = iz < G.nz;

    // this lane's slab: rows with non-zero weight, in row order (k_sf_bp skips
    // the zero weights, and the whole view when the slab meets no row)
    SlabWeights SW;
    par3_slab_rows(G, zin ? iz : 0, SW);
    int nzr = 0, rq[kSlabs];
    float rw[kSlabs];
#pragma unroll
    for (int q = 0; q < kSlabs; ++q) {
        rq[q] = 0;
        rw[q] = 0.0f;
    }
#pragma unroll
    for (int q = 0; q < kSlabs; ++q) {
        if (SW.w[q] > 0.0f) {
#pragma unroll
            for (int s = 0; s < kSlabs; ++s) {  // slot nzr, without dynamic register indexing
                if (s == nzr) {
                    rq[s] = SW.first + q;
                    rw[s] = SW.w[q];
                }
            }
            ++nzr;
        }
    }
    if (!zin || SW.count <= 0) nzr = 0;

    // rows any lane of the wave needs per bin (wave-uniform)
    int nzr_max = nzr;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) nzr_max = max(nzr_max, __shfl_xor(nzr_max, m));
    const int nzr_u = __builtin_amdgcn_readfirstlane(nzr_max);
    const bool pre = nzr_u <= 2;

    const float u0 = sf_det(G.nu, G.du, G.su, 0);
    const float inv_du = 1.0f / G.du;
    const float* sb = sino + (int64_t)b * G.na * G.nu * G.nv;
    double acc = 0.0;
    // the view loop, for NR preloaded rows per bin: one where no slab of the
    // wave meets a second row (rows aligned with the slabs), else two
    auto views = [&](auto nr_tag) {
        constexpr int NR = decltype(nr_tag)::value;
        for (int va = 0; va < G.na; va += 64) {
            // lane = view va + lane: bins of this pixel's footprint with positive overlap
            int cnt = 0, jl[kJMax];
            float wl[kJMax];
#pragma unroll
            for (int s = 0; s < kJMax; ++s) {
                jl[s] = 0;
                wl[s] = 0.0f;
            }
            const int ial = va + lane;
            if (ial < G.na) {
                const SFView V = sf_view(G, cs[ial], sn[ial], ang[ial]);
                const SFFoot f = sf_foot<SF_PAR3>(G, V, ix, iy);
                if (f.u1 > u0 - G.du && (f.u0 - u0) * inv_du < (float)G.nu + 1.0f) {
                    const int j0 = (int)fmaxf(floorf((f.u0 - u0) * inv_du) - 1.0f, 0.0f);
                    const int j1 = (int)fminf(floorf((f.u1 - u0) * inv_du) + 1.0f, (float)(G.nu - 1));
#pragma unroll
                    for (int t = 0; t < kJMax; ++t) {
                        const int j = j0 + t;
                        if (j > j1) break;
                        const float ou = ovl(f.u0, f.u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
                        if (!(ou > 0.0f)) continue;
                        const float wu = (ou * inv_du) * f.amp;
#pragma unroll
                        for (int s = 0; s < kJMax; ++s) {
                            if (s == cnt) {
                                jl[s] = j;
                                wl[s] = wu;
                            }
                        }
                        ++cnt;
                    }
                }
            }
            const int nvw = min(64, G.na - va);
            for (int v = 0; v < nvw; ++v) {
                const int c = __builtin_amdgcn_readlane(cnt, v);
                const float* plane = sb + (int64_t)(va + v) * G.nu * G.nv;
                // the rows of the first kJPre bins, two per slab, are loaded
                // together before any is used, by every lane and for every one
                // of these bins: bins past the footprint's count read bin jl = 0,
                // rows past the slab's count row rq = 0, both valid, and the sums
                // below skip them
                float xv[kJPre][2];
                if (pre) {
#pragma unroll
                    for (int s = 0; s < kJPre; ++s) {
                        const float* row = plane + (int64_t)__builtin_amdgcn_readlane(jl[s], v) * G.nv;
                        xv[s][0] = row[rq[0]];
                        xv[s][1] = NR > 1 ? row[rq[1]] : 0.0f;
                    }
                }
#pragma unroll
                for (int s = 0; s < kJMax; ++s) {
                    if (s >= c) break;
                    const float wu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl[s]), v));
                    float sv_ = 0.0f;
                    if (s < kJPre && pre) {
                        const int sp = s < kJPre ? s : 0;
                        sv_ = 0 < nzr ? sv_ + xv[sp][0] * rw[0] : sv_;
                        if (NR > 1) sv_ = 1 < nzr ? sv_ + xv[sp][1] * rw[1] : sv_;
                    } else {
                        const int j = __builtin_amdgcn_readlane(jl[s], v);
                        const float* row = plane + (int64_t)j * G.nv;
#pragma unroll
                        for (int q = 0; q < kSlabs; ++q)
                            if (q < nzr) sv_ += row[rq[q]] * rw[q];
                    }
                    acc = __builtin_fma((double)wu, (double)sv_, acc);
                }
            }
        }
    };
    if (nzr_u <= 1)
        views(std::integral_constant<int, 1>{});
    else
        views(std::integral_constant<int, 2>{});
    if (!zin) return;
    const int64_t o = (((int64_t)b * G.nx + ix) * G.ny + iy) * G.nz + iz;
    float res = (float)acc * G.out_scale;
    if (accumulate) res += img[o];
    img[o] = res;
}

// ------------------------------- parallel 3-D backward on the matrix cores
//
// Rows aligned with the slabs (slab z meets row z + shift only): a block of 4 x
// 4 pixels backprojects a view as the product of its 16 x 4 KS footprint
// weights and 4 KS sinogram rows, in float64 (v_mfma_f64_16x16x4_f64: exact
// products of the float32 weights and values, float64 sums).  A lane evaluates
// the weights that its operand slot needs -- pixel lane % 16, bin jb + 4 kk +
// lane / 16 -- so there are no lists and no broadcasts, and a row is read once
// for sixteen pixels.  Four accumulators cover 64 slabs.  The column kernel
// above spends 184 cycles a pixel column and view on broadcasts, loads and sums
// (7.0 ms for 8 x 256 x 256 x 64, 180 views of 384); this one 55 (2.1 ms), of
// which 36 are the product's, a third of it on non-zero weights.
//
// Zero weights times infinite values make NaNs: where a sum is not finite, the
// wave's pixels are done again bin by bin.
typedef double sf_d4 __attribute__((ext_vector_type(4)));

// One voxel (pixel (ix, iy), row m, weight rw of its slab) by the gather.
__device__ double sf_bp_par3_one(const SFGeo& G, const float* __restrict__ cs, const float* __restrict__ sn,
                                 const float* __restrict__ sb, int ix, int iy, int m, float rw) {
    double acc = 0.0;
    if (!(rw > 0.0f)) return acc;
    const float u0 = sf_det(G.nu, G.du, G.su, 0), inv_du = 1.0f / G.du;
    for (int ia = 0; ia < G.na; ++ia) {
        const SFView V = sf_view(G, cs[ia], sn[ia], 0.0f);
        const SFFoot f = sf_foot<SF_PAR3>(G, V, ix, iy);
        if (!(f.u1 > u0 - G.du) || !((f.u0 - u0) * inv_du < (float)G.nu + 1.0f)) continue;
        const int j0 = (int)fmaxf(floorf((f.u0 - u0) * inv_du) - 1.0f, 0.0f);
        const int j1 = (int)fminf(floorf((f.u1 - u0) * inv_du) + 1.0f, (float)(G.nu - 1));
        for (int j = j0; j <= j1; ++j) {
            const float ou = ovl(f.u0, f.u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
            if (ou > 0.0f)
                acc = __builtin_fma((double)((ou * inv_du) * f.amp),
                                    (double)(sb[((int64_t)ia * G.nu + j) * G.nv + m] * rw), acc);
        }
    }
    return acc;
}

// SPLIT: the four waves of a block share one pixel block's views (few blocks)
// and add their sums in wave order; else each takes a block of its own.
template <int KS, bool SPLIT>
__global__ __launch_bounds__(256) void k_sf_bp_par3_mfma(SFGeo G, const float* __restrict__ cs,
                                                        const float* __restrict__ sn,
                                                        const float* __restrict__ sino, float* __restrict__ img,
                                                        int accumulate, int nby, int nbx, int nzt, int shift,
                                                        int64_t nblk) {
    __shared__ double red[SPLIT ? 4 : 1][SPLIT ? 1024 : 1];
    const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t blk = xcd_remap(blockIdx.x, gridDim.x);
    int64_t wid = SPLIT ? blk : blk * 4 + wave;
    if (wid >= nblk) return;  // whole wave (SPLIT: whole block)
    const int zb = (int)(wid % nzt) * 64;
    wid /= nzt;
    const int by = (int)(wid % nby) * 4;
    wid /= nby;
    const int bx = (int)(wid % nbx) * 4;
    const int b = (int)(wid / nbx);
    const float* __restrict__ sb = sino + (int64_t)b * G.na * G.nu * G.nv;
    const float inv_du = 1.0f / G.du, inv_dv = 1.0f / G.dv, half = 0.5f * (float)G.nu;
    // slabs z = zb + 16 zg + lo: their row and its weight
    const int nzg = min(4, (G.nz - zb + 15) / 16);
    int off[4];
    float rw[4];
#pragma unroll
    for (int zg = 0; zg < 4; ++zg) {
        const int z = zb + 16 * zg + lo, m = z + shift;
        off[zg] = hi * G.nv + min(max(m, 0), G.nv - 1);
        const float ov = sf_bnd(G.nz, G.d, z + 1) - sf_bnd(G.nz, G.d, z);
        rw[zg] = z < G.nz && m >= 0 && m < G.nv ? ov * inv_dv : 0.0f;
    }
    // weights: pixel (bx + lo / 4, by + lo % 4)
    const float xc = G.d * (((float)(bx + (lo >> 2)) + 0.5f) - 0.5f * (float)G.nx);
    const float yc = G.d * (((float)(by + (lo & 3)) + 0.5f) - 0.5f * (float)G.ny);
    const float xm = G.d * ((float)(bx + 2) - 0.5f * (float)G.nx), ym = G.d * ((float)(by + 2) - 0.5f * (float)G.ny);
    const float eps = 0.01f + 1e-6f * (float)G.nu;
    sf_d4 acc[4];
#pragma unroll
    for (int zg = 0; zg < 4; ++zg) acc[zg] = sf_d4{0.0, 0.0, 0.0, 0.0};
    const int vstep = SPLIT ? 4 : 1, vfirst = SPLIT ? wave : 0;
    for (int g = vfirst; g < G.na; g += 64 * vstep) {
        // lane = view g + vstep lane: its constants and the block's first bin
        const int il = min(g + vstep * lane, G.na - 1);
        const SFView L = sf_view(G, cs[il], sn[il], 0.0f);
        const float lf = (-L.s * xm + L.c * ym - 4.0f * L.h) * inv_du - G.su + half;
        const int jl = (int)fminf(fmaxf(floorf(lf - eps), 0.0f), (float)(G.nu - 4 * KS));
        const int nl = min(64, (G.na - g + vstep - 1) / vstep);
        struct View {
            float x[KS][4];
            double w[KS];
        };
        const auto load = [&](int l, View& T) {
            const float c = ct_lane(L.c, l), s = ct_lane(L.s, l), amp = ct_lane(L.amp, l), h = ct_lane(L.h, l);
            const int jb = __builtin_amdgcn_readlane(jl, l);
            const float* __restrict__ p = sb + ((int64_t)(g + vstep * l) * G.nu + jb) * G.nv;
#pragma unroll
            for (int kk = 0; kk < KS; ++kk)
#pragma unroll
                for (int zg = 0; zg < 4; ++zg)
                    if (zg < nzg) T.x[kk][zg] = p[(int64_t)4 * kk * G.nv + off[zg]];
            const float pc = -s * xc + c * yc, u0 = pc - h, u1 = pc + h;
#pragma unroll
            for (int kk = 0; kk < KS; ++kk) {
                const int j = jb + 4 * kk + hi;
                const float ou = ovl(u0, u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
                T.w[kk] = ou > 0.0f && h < VIR_INF ? (double)((ou * inv_du) * amp) : 0.0;
            }
        };
        const auto use = [&](const View& T) {
#pragma unroll
            for (int kk = 0; kk < KS; ++kk)
#pragma unroll
                for (int zg = 0; zg < 4; ++zg)
                    if (zg < nzg)
                        acc[zg] = __builtin_amdgcn_mfma_f64_16x16x4f64(T.w[kk], (double)(T.x[kk][zg] * rw[zg]), acc[zg],
                                                                       0, 0, 0);
        };
        // the next view's rows are on their way while a view is multiplied
        View A, B;
        load(0, A);
        for (int l = 0; l < nl; l += 2) {
            if (l + 1 < nl) load(l + 1, B);
            use(A);
            if (l + 1 >= nl) break;
            if (l + 2 < nl) load(l + 2, A);
            use(B);
        }
    }
    // element r of acc[zg]: pixel (bx + r, by + hi), slab zb + 16 zg + lo
    if (SPLIT) {
#pragma unroll
        for (int zg = 0; zg < 4; ++zg)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][256 * zg + 64 * r + lane] = acc[zg][r];
        __syncthreads();
    }
#pragma unroll
    for (int zg = 0; zg < 4; ++zg) {
        if (zg >= nzg || (SPLIT && zg != wave)) continue;
        sf_d4 v = acc[zg];
        if constexpr (SPLIT) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = 256 * zg + 64 * r + lane;
                v[r] = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
            }
        }
        const int z = zb + 16 * zg + lo;
        const bool bad = !(fabs(v[0]) + fabs(v[1]) + fabs(v[2]) + fabs(v[3]) < (double)VIR_INF);
        const bool again = __any(bad);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int ix = bx + r, iy = by + hi;
            if (ix >= G.nx || iy >= G.ny || z >= G.nz) continue;
            if (again) v[r] = sf_bp_par3_one(G, cs, sn, sb, ix, iy, min(max(z + shift, 0), G.nv - 1), rw[zg]);
            const int64_t o = (((int64_t)b * G.nx + ix) * G.ny + iy) * G.nz + z;
            float res = (float)v[r] * G.out_scale;
            if (accumulate) res += img[o];
            img[o] = res;
        }
    }
}

// K-steps of the matrix backprojector for the geometry (a 4 x 4 pixel block is
// at most 4 sqrt(2) d wide on the detector: that many bins and two), or 0 where
// it does not apply: rows not aligned with the slabs, footprints too wide, a
// detector narrower than a block's window.
static int sf_par3_bp_ksteps(const SFGeo& G, int& shift) {
    const double t = 0.5 * ((double)G.nv - G.nz) - (double)G.sv;
    if (G.dv != G.d || t != std::floor(t) || std::fabs(t) > 1e6 || G.nu > 15000) return 0;  // (eps: 0.025 bin)
    shift = (int)t;
    const int ks = ((int)std::floor(4.0 * 1.41422 * (double)G.d / (double)G.du + 0.05) + 2 + 3) / 4;
    return ks <= 4 && G.nu >= 4 * ks ? ks : 0;
}

// Items of fewer pixel blocks split each one's views over four waves.  Split |
// one wave a block, us: 256 x 256 x 64 (4096 blocks), 180 views, one item 277 | 294,
// eight 2102 | 2038, 45 views 78 | 77, 583 | 527; 128 x 128 x 64 (1024 blocks), 180
// views, 32 items 2135 | 2056, one 76 | (too few waves).
constexpr int64_t kParSplit = 4096;

template <int KS>
static int sf_par3_bp_mfma(const SFGeo& G, const float* cosv, const float* sinv, const float* sino, float* img, int acc,
                           int shift, hipStream_t st) {
    const int nbx = (G.nx + 3) / 4, nby = (G.ny + 3) / 4, nzt = (G.nz + 63) / 64;
    const int64_t n = (int64_t)G.nb * nbx * nby * nzt;
    // by one item's blocks, so that an item's bits don't depend on the batch
    if ((int64_t)nbx * nby * nzt < kParSplit)
        hipLaunchKernelGGL((k_sf_bp_par3_mfma<KS, true>), dim3((unsigned)n), dim3(256), 0, st, G, cosv, sinv, sino, img,
                           acc, nby, nbx, nzt, shift, n);
    else
        hipLaunchKernelGGL((k_sf_bp_par3_mfma<KS, false>), dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, G, cosv, sinv,
                           sino, img, acc, nby, nbx, nzt, shift, n);
    return check_hip(hipGetLastError(), "vir_sf_bp launch");
}

// True when the column backprojector applies: a slab meets at most kSlabs
// detector rows (rows at least half a voxel tall) and a pixel footprint at
// most kJMax bins.
static bool sf_par3_bp_col_ok(const SFGeo& G) {
    if (!((double)G.d / (double)G.dv <= 1.99)) return false;
    return 1.4143 * (double)G.d / (double)G.du + 4.0 <= (double)kJMax;
}

// True when the tiled parallel 3-D forward kernel takes the call: detector rows
// no taller than a voxel (each row meets at most kSlabs slabs), and where it is
// faster than the gather, judged by one item so that an item's bits don't depend
// on the batch.  256 x 256, 1.5 x 256 bins, tile | gather in us, 8 items, 180
// views, 64 rows: du = d 2930 | 28500, 2 d 2980 | 17600; 1 item, 64 views: 500 |
// 1635, 1140 | 1230.  8 items with 4 rows 2910 | 2225, with 8: 2910 | 3910; 1 item,
// 64 views, 4 rows 500 | 480.
// Bins wider than 2.5 pixels have long pixel windows, and a block takes its 1.5
// ms at 256^2 however few there are.  An item needs blocks (counted by the rows
// in use) to make up for it: below 2.75 pixels as many as let a batch fill
// the chip, from 2.75 on as many as win alone.  2.6 | 2.8 | 3.2 | 4 pixels, gather
// over tile, 64 rows: 450 | 405 | 360 | 270 blocks, one item 1.58 | 1.61 | 1.34 | 0.82,
// eight 4.4 | 4.0 | 3.5 | 2.9; 160 | 144 | 128 | 96: 0.89 | 0.78 | 0.74 | 0.55, 2.9 | 2.6 |
// 2.2 | 1.8; 48 | 48 | 32 | 32: 0.66 | 0.65 | 0.69 | 0.52, 1.8 | 1.5 | 1.6 | 1.1; 20 | 20 | 16 |
// 12: 0.51 | 0.52 | 0.51 | 0.40, 1.0 | 1.0 | 0.9 | 0.7.
static bool sf_par3_tiled_ok(const SFGeo& G) {
    if (!(G.dv <= G.d) || G.nv < 6) return false;
    if (G.du <= 2.5f * G.d) return true;
    const double full = (double)((G.na + kVG - 1) / kVG) * ((G.nu + kTUB - 1) / kTUB) * G.nv / kTV;
    return G.du <= 2.75f * G.d ? full >= 48.0 : G.du <= 3.2f * G.d && full >= 350.0;
}

// An item with at most this many blocks (two a CU) takes two wave groups a
// block: they wait for their own chain of operands, not for the matrix cores.
// 256 x 256 x 64, 64 views (384 blocks) 682 -> 500 us; with 8 items and 180 views
// (8640 blocks) one group is the faster one, 2940 against 3660 us.
constexpr int kParBlocks2 = 512;

// True when every row m meets slab m - shift alone with weight 1: rows aligned
// with the slabs, and a power-of-two spacing, so that overlap / dv is exact.
static bool sf_par3_unit_rows(const SFGeo& G, int& shift) {
    const double t = 0.5 * ((double)G.nv - G.nz) - (double)G.sv;
    int e;
    if (G.dv != G.d || t != std::floor(t) || std::fabs(t) > 1e6 || std::frexp(G.d, &e) != 0.5f) return false;
    shift = (int)t;
    return true;
}

template <int MODE>
__global__ __launch_bounds__(256) void k_sf_bp(SFGeo G, const float* __restrict__ ang,
                                              const float* __restrict__ cs, const float* __restrict__ sn,
                                              const float* __restrict__ sino, float* __restrict__ img,
                                              int accumulate) {
    const bool is3 = MODE == SF_CONE3 || MODE == SF_PAR3;
    const int nz = is3 ? G.nz : 1, nv = is3 ? G.nv : 1;
    const int64_t per_b = (int64_t)G.nx * G.ny * nz;
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= per_b * G.nb) return;
    const int b = (int)(t / per_b);
    int64_t r = t % per_b;
    const int iz = (int)(r % nz);
    const int iy = (int)((r / nz) % G.ny);
    const int ix = (int)(r / ((int64_t)nz * G.ny));
    const float u0 = sf_det(G.nu, G.du, G.su, 0), v0 = sf_det(nv, G.dv, G.sv, 0);
    const float inv_du = 1.0f / G.du, inv_dv = 1.0f / G.dv;
    const float zl = sf_bnd(G.nz, G.d, iz), zr = sf_bnd(G.nz, G.d, iz + 1);
    const float* sb = sino + (int64_t)b * G.na * G.nu * nv;
    // parallel 3-D: the detector rows this slab meets and their weights
    SlabWeights SW;
    SW.first = 0;
    SW.count = 0;
    bool row_general = false;
    if (MODE == SF_PAR3) row_general = !par3_slab_rows(G, iz, SW);
    double acc = 0.0;
    for (int ia = 0; ia < G.na; ++ia) {
        const SFView V = sf_view(G, cs[ia], sn[ia], ang[ia]);
        const SFFoot f = sf_foot<MODE>(G, V, ix, iy);
        if (!(f.u1 > u0 - G.du) || !((f.u0 - u0) * inv_du < (float)G.nu + 1.0f)) continue;
        int j0 = (int)fmaxf(floorf((f.u0 - u0) * inv_du) - 1.0f, 0.0f);
        int j1 = (int)fminf(floorf((f.u1 - u0) * inv_du) + 1.0f, (float)(G.nu - 1));
        const float* plane = sb + (int64_t)ia * G.nu * nv;
        if (!is3) {
            for (int j = j0; j <= j1; ++j) {
                const float ou = ovl(f.u0, f.u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
                if (ou > 0.0f) acc += (double)(plane[j] * ((ou * inv_du) * f.amp));
            }
            continue;
        }
        if (MODE == SF_PAR3 && !row_general) {
            if (SW.count <= 0) continue;
            for (int j = j0; j <= j1; ++j) {
                const float ou = ovl(f.u0, f.u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
                if (!(ou > 0.0f)) continue;
                const float wu = (ou * inv_du) * f.amp;
                const float* rowp = plane + (int64_t)j * nv + SW.first;
                float sv_ = 0.0f;
#pragma unroll
                for (int q = 0; q < kSlabs; ++q)
                    if (SW.w[q] > 0.0f) sv_ += rowp[q] * SW.w[q];
                acc = __builtin_fma((double)wu, (double)sv_, acc);
            }
            continue;
        }
        float qa = f.cm * zl, qb = f.cm * zr;
        float lo = fminf(qa, qb), hi = fmaxf(qa, qb);
        if (!(hi > v0 - G.dv) || !((lo - v0) * inv_dv < (float)nv + 1.0f)) continue;
        int m0 = (int)fmaxf(floorf((lo - v0) * inv_dv) - 1.0f, 0.0f);
        int m1 = (int)fminf(floorf((hi - v0) * inv_dv) + 1.0f, (float)(nv - 1));
        for (int j = j0; j <= j1; ++j) {
            const float ou = ovl(f.u0, f.u1, sf_det(G.nu, G.du, G.su, j), sf_det(G.nu, G.du, G.su, j + 1));
            if (!(ou > 0.0f)) continue;
            const float wu = (ou * inv_du) * f.amp;
            for (int m = m0; m <= m1; ++m) {
                float ov = ovl(qa, qb, sf_det(nv, G.dv, G.sv, m), sf_det(nv, G.dv, G.sv, m + 1));
                if (ov > 0.0f) acc += (double)(plane[(int64_t)j * nv + m] * (wu * (ov * inv_dv)));
            }
        }
    }
    float res = (float)acc * G.out_scale;
    if (accumulate) res += img[t];
    img[t] = res;
}

// Slabs a detector row (forward) or rows a slab (backward) of the cone
// geometry can meet, from the magnifications at the grid's rim (times 1/cos of
// the largest fan angle, tan <= R/sqrt(DSO^2 - R^2)); 0: the tiles do not apply or
// do not pay.
static int sf_cone_slots(const SFGeo& G, bool fp, uint32_t flags) {
    if (flags & VIR_PER_OUTPUT) return 0;
    const double R = 0.5 * std::sqrt((double)G.nx * G.nx + (double)G.ny * G.ny) * G.d, D = G.DSO;
    if (fp && ct_few_rows(G)) return 0;
    return fp ? ct_slots((double)G.dv * (D + R) / ((double)G.DSD * G.d), G.nz)
              : ct_slots((double)G.d * G.DSD / (D - R) * (D / std::sqrt(D * D - R * R)) / G.dv, G.nv);
}

// Threads that one item's launch takes (at most; fewer in a batch of many).
static int64_t sf_threads(const SFGeo& G, int mode, bool fp) {
    if (mode == SF_PAR2 || mode == SF_FAN2) return ft_threads(G, fp);
    if (mode == SF_CONE3) return ct_threads(G, fp);
    if (fp) {
        const int64_t n = (int64_t)((G.na + kVG - 1) / kVG) * ((G.nu + kTUB - 1) / kTUB) * ((G.nv + kTV - 1) / kTV);
        return n * 64 * kVG * (n <= kParBlocks2 ? 2 : 1);
    }
    int shift;
    const int64_t nzt = (G.nz + 63) / 64, n = (int64_t)((G.nx + 3) / 4) * ((G.ny + 3) / 4) * nzt;
    return sf_par3_bp_ksteps(G, shift) ? n * (n < kParSplit ? 256 : 64) + 256 : (int64_t)G.nx * G.ny * nzt * 64 + 256;
}

// A batch in parts, where a launch can't have the threads of all items (items
// don't depend on their batch); flags gets VIR_PER_OUTPUT where it can't have
// those of one.
template <class Call>
static int sf_parts(const vir_sf_geom* geom, const SFGeo& G, bool fp, const float* src, float* dst, uint32_t& flags,
                    Call&& call, bool& done) {
    done = false;
    if (flags & VIR_PER_OUTPUT) return VIR_OK;
    const int64_t per = sf_threads(G, geom->mode, fp);
    if (per > kLaunchThreads) {
        flags |= VIR_PER_OUTPUT;
        return VIR_OK;
    }
    const int64_t most = kLaunchThreads / per;
    if (G.nb <= most) return VIR_OK;
    done = true;
    const int64_t vox = (int64_t)G.nx * G.ny * G.nz, bins = (int64_t)G.na * G.nu * G.nv;
    for (int64_t b = 0; b < G.nb; b += most) {
        vir_sf_geom g = *geom;
        g.nbatch = (int32_t)std::min<int64_t>(most, G.nb - b);
        if (const int rc = call(&g, src + b * (fp ? vox : bins), dst + b * (fp ? bins : vox))) return rc;
    }
    return VIR_OK;
}

static int sf_setup(const vir_sf_geom* g, SFGeo& G) {
    if (!g) return fail_arg("geometry is NULL");
    if (g->mode < 0 || g->mode > 3) return fail_arg("mode must be 0..3");
    bool is3 = g->mode == SF_CONE3 || g->mode == SF_PAR3;
    G.nx = g->nx; G.ny = g->ny; G.nz = is3 ? g->nz : 1;
    G.nu = g->nu; G.nv = is3 ? g->nv : 1; G.na = g->na; G.nb = g->nbatch;
    G.d = g->d_pix; G.du = g->du; G.dv = is3 ? g->dv : 1.0f;
    G.su = g->su; G.sv = is3 ? g->sv : 0.0f; G.DSO = g->DSO; G.DSD = g->DSD;
    G.out_scale = 1.0f;
    G.unit_amp = 0;
    G.compat = 0;
    if (G.nx < 1 || G.ny < 1 || G.nz < 1 || G.nu < 1 || G.nv < 1 || G.na < 0 || G.nb < 1)
        return fail_arg("bad sizes");
    if (!(G.d > 0.0f) || !(G.du > 0.0f) || !(G.dv > 0.0f)) return fail_arg("spacings must be > 0");
    // Largest distance between a pixel's centre projection and any point of
    // its footprint (the footprint contains the centre projection):
    //   parallel: half the projected diagonal, d/sqrt(2);
    //   fan/cone: a corner offset (dp, do) from the centre moves the
    //   projection by DSD*(dp + t*do)/(DSO - o_corner) with t = u_c/DSD, so
    //   the distance is at most mag * (d/sqrt(2)) * sqrt(1 + t^2), where
    //   mag = DSD/(DSO - R) and |t| <= R/sqrt(DSO^2 - R^2) over the disc of
    //   radius R (the grid's half-diagonal) that holds every pixel.
    const double hx = 0.5 * G.nx * (double)G.d, hy = 0.5 * G.ny * (double)G.d;
    const double R = std::sqrt(hx * hx + hy * hy);
    double w = (double)G.d * 0.70710678118654752;
    if (g->mode == SF_FAN2 || g->mode == SF_CONE3) {
        if (!(G.DSO > 0.0f) || !(G.DSD > 0.0f)) return fail_arg("DSO and DSD must be > 0");
        if (!(R < 0.999 * G.DSO)) return fail_arg("grid reaches the source (DSO too small)");
        const double D = G.DSO;
        w *= (double)G.DSD / (D - R) * (D / std::sqrt(D * D - R * R));
    }
    G.wmax = (float)(1.02 * w + 1e-3 * (double)G.du);
    if (g->mode == SF_FAN2 || g->mode == SF_CONE3) {
        // the forward gather inverts the centre projection along the driving
        // axis; that inverse is monotone while |u| < DSD (fan half-angle
        // below 45 degrees), so the detector plus margin must stay inside
        const double umax = (double)G.du * std::fmax(std::fabs(-0.5 * G.nu + G.su),
                                                     std::fabs(0.5 * G.nu + G.su)) + G.wmax;
        if (!(umax < 0.999 * (double)G.DSD))
            return fail_arg("detector reaches a 45 degree fan half-angle (|u| >= DSD)");
    }
    return VIR_OK;
}

}  // namespace vir

using namespace vir;

// Small images on detectors a fraction of the 2-D tile's 128 bins wide: with rows
// enough to fill the chip one thread per bin is faster.  (Lines the tile stages at
// once, so both give the same bits and the batch may count.)  Tile | per output, us:
// parallel 16^2, 11520 rows of 24 bins 53 | 40, of 48 53 | 60, 92160 rows of 24 356 | 182;
// 64^2, 128000 rows of 33 bins 1895 | 1570, of 48 1718 | 2006; fan 64^2, 128000 rows of 16
// bins 8908 | 6700, of 24 8203 | 8190.
static bool sf_narrow(const SFGeo& G, int mode) {
    const int64_t rows = (int64_t)G.nb * G.na;
    return std::max(G.nx, G.ny) <= 64 && (mode == SF_PAR2 ? G.nu <= 36 && rows >= 8192 : G.nu <= 20 && rows >= 50000);
}

extern "C" {

int vir_sf_fp(const vir_sf_geom* geom, const float* ang, const float* cosv, const float* sinv, const float* img,
              float* sino, float out_scale, uint32_t flags, void* stream) {
    SFGeo G;
    int rc = sf_setup(geom, G);
    if (rc) return rc;
    if (G.na == 0) return VIR_OK;
    if (!ang || !cosv || !sinv || !img || !sino) return fail_arg("NULL pointer argument");
    G.out_scale = out_scale;
    G.unit_amp = (flags & VIR_SF_UNIT_AMPLITUDE) ? 1 : 0;
    G.compat = (flags & VIR_COMPAT) ? 1 : 0;
    bool done;
    const uint32_t given = flags;
    rc = sf_parts(geom, G, true, img, sino, flags, [&](const vir_sf_geom* g, const float* src, float* dst) {
        return vir_sf_fp(g, ang, cosv, sinv, src, dst, out_scale, given, stream);
    }, done);
    if (rc || done) return rc;
    int64_t n = (int64_t)G.nb * G.na * G.nu * G.nv;
    dim3 grd((unsigned)((n + 255) / 256));
    hipStream_t st = as_stream(stream);
    int acc = (flags & VIR_ACCUMULATE) ? 1 : 0;
    // VIR_COMPAT's amplitudes depend on the pixels before: the gather looks back
    const bool flat = !G.compat && !(flags & VIR_PER_OUTPUT) && !sf_narrow(G, geom->mode);
    if (flat && geom->mode == SF_PAR2)
        return ft_fp<SFFlat<SF_PAR2>>(G, G.nb, ang, cosv, sinv, img, sino, acc, st, SirtEpi{}, "vir_sf_fp launch");
    if (flat && geom->mode == SF_FAN2)
        return ft_fp<SFFlat<SF_FAN2>>(G, G.nb, ang, cosv, sinv, img, sino, acc, st, SirtEpi{}, "vir_sf_fp launch");
    switch (geom->mode) {
        case SF_PAR2: hipLaunchKernelGGL(k_sf_fp<SF_PAR2>, grd, dim3(256), 0, st, G, ang, cosv, sinv, img, sino, acc); break;
        case SF_FAN2: hipLaunchKernelGGL(k_sf_fp<SF_FAN2>, grd, dim3(256), 0, st, G, ang, cosv, sinv, img, sino, acc); break;
        case SF_CONE3:
            if (const int ns = sf_cone_slots(G, true, flags))
                return ct_fp<SFCone>(G, G.nb, ns, ang, cosv, sinv, img, sino, acc, st, "vir_sf_fp launch");
            hipLaunchKernelGGL(k_sf_fp<SF_CONE3>, grd, dim3(256), 0, st, G, ang, cosv, sinv, img, sino, acc); break;
        default:
            if (sf_par3_tiled_ok(G) && !(flags & VIR_PER_OUTPUT)) {
                const int nut = (G.nu + kTUB - 1) / kTUB, nmt = (G.nv + kTV - 1) / kTV;
                const int nvg = (G.na + kVG - 1) / kVG;
                const dim3 tg((unsigned)((int64_t)G.nb * nvg * nut * nmt));
                int shift = 0;
                const bool unit = sf_par3_unit_rows(G, shift);
                // by one item's blocks, so that an item's bits don't depend on the batch
                const bool two = nvg * nut * nmt <= kParBlocks2;
                const auto kern = unit ? (two ? k_sf_fp_par3_mfma<true, 2> : k_sf_fp_par3_mfma<true, 1>)
                                       : (two ? k_sf_fp_par3_mfma<false, 2> : k_sf_fp_par3_mfma<false, 1>);
                hipLaunchKernelGGL(kern, tg, dim3(64 * kVG * (two ? 2 : 1)), 0, st, G, cosv, sinv, img, sino, acc, nut,
                                   nmt, nvg, shift);
            } else {
                hipLaunchKernelGGL(k_sf_fp<SF_PAR3>, grd, dim3(256), 0, st, G, ang, cosv, sinv, img, sino, acc);
            }
            break;
    }
    return check_hip(hipGetLastError(), "vir_sf_fp launch");
}

int vir_sf_bp(const vir_sf_geom* geom, const float* ang, const float* cosv, const float* sinv, const float* sino,
              float* img, float out_scale, uint32_t flags, void* stream) {
    SFGeo G;
    int rc = sf_setup(geom, G);
    if (rc) return rc;
    if ((G.na > 0 && (!ang || !cosv || !sinv || !sino)) || !img) return fail_arg("NULL pointer argument");
    G.out_scale = out_scale;
    G.unit_amp = (flags & VIR_SF_UNIT_AMPLITUDE) ? 1 : 0;
    bool done;
    const uint32_t given = flags;
    rc = sf_parts(geom, G, false, sino, img, flags, [&](const vir_sf_geom* g, const float* src, float* dst) {
        return vir_sf_bp(g, ang, cosv, sinv, src, dst, out_scale, given, stream);
    }, done);
    if (rc || done) return rc;
    int64_t n = (int64_t)G.nb * G.nx * G.ny * G.nz;
    dim3 grd((unsigned)((n + 255) / 256));
    hipStream_t st = as_stream(stream);
    int acc = (flags & VIR_ACCUMULATE) ? 1 : 0;
    const bool flat = !(flags & VIR_PER_OUTPUT);
    if (flat && geom->mode == SF_PAR2)
        return ft_bp<SFFlat<SF_PAR2>>(G, G.nb, ang, cosv, sinv, sino, img, acc, st, SirtEpi{}, "vir_sf_bp launch");
    if (flat && geom->mode == SF_FAN2)
        return ft_bp<SFFlat<SF_FAN2>>(G, G.nb, ang, cosv, sinv, sino, img, acc, st, SirtEpi{}, "vir_sf_bp launch");
    switch (geom->mode) {
        case SF_PAR2: hipLaunchKernelGGL(k_sf_bp<SF_PAR2>, grd, dim3(256), 0, st, G, ang, cosv, sinv, sino, img, acc); break;
        case SF_FAN2: hipLaunchKernelGGL(k_sf_bp<SF_FAN2>, grd, dim3(256), 0, st, G, ang, cosv, sinv, sino, img, acc); break;
        case SF_CONE3:
            if (const int ns = sf_cone_slots(G, false, flags))
                return ct_bp<SFCone>(G, G.nb, ns, ang, cosv, sinv, sino, img, acc, st, "vir_sf_bp launch");
            hipLaunchKernelGGL(k_sf_bp<SF_CONE3>, grd, dim3(256), 0, st, G, ang, cosv, sinv, sino, img, acc); break;
        default:
            if (int shift = 0; !(flags & VIR_PER_OUTPUT)) {
                const int ks = sf_par3_bp_ksteps(G, shift);
                if (ks == 1) return sf_par3_bp_mfma<1>(G, cosv, sinv, sino, img, acc, shift, st);
                if (ks == 2) return sf_par3_bp_mfma<2>(G, cosv, sinv, sino, img, acc, shift, st);
                if (ks == 3) return sf_par3_bp_mfma<3>(G, cosv, sinv, sino, img, acc, shift, st);
                if (ks == 4) return sf_par3_bp_mfma<4>(G, cosv, sinv, sino, img, acc, shift, st);
            }
            if (sf_par3_bp_col_ok(G) && !(flags & VIR_PER_OUTPUT)) {
                const int nzt = (G.nz + 63) / 64;
                const int64_t nw = (int64_t)G.nb * G.nx * G.ny * nzt;
                hipLaunchKernelGGL(k_sf_bp_par3_col, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0, st, G, ang, cosv,
                                   sinv, sino, img, acc, nzt);
            } else {
                hipLaunchKernelGGL(k_sf_bp<SF_PAR3>, grd, dim3(256), 0, st, G, ang, cosv, sinv, sino, img, acc);
            }
            break;
    }
    return check_hip(hipGetLastError(), "vir_sf_bp launch");
}

}  // extern "C"
