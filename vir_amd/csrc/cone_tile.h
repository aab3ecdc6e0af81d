// Cone-beam footprint projections in tiles, shared by the distance-driven
// (dd.hip) and separable-footprint (sf.hip) projectors.
//
// Both models weigh voxel (pixel, slab) on detector bin (u, v) by
//   w(pixel, u) * |slab's magnified z interval  n  row v|,
// separable in u and v but for the z magnification, which depends on the
// pixel (separable footprint) or on its line only (distance driven).  A model
// M gives, per view:
//   M(G, c, s, ang)                    the view
//   xd, nd, no                         driving axis, pixels a line, lines
//   range(lo, hi, io, k0, k1)          pixels of line io that can meet the bin
//                                      edges [lo, hi] (false: none)
//   weight(k, io, lo, hi)              w of pixel k for those edges, <= 0: none
//   zmag(k, io)                        z magnification
//   foot(k, io, lo, hi)                the pixel's interval along u
//   fp_unit(G), bp_unit(G)             factors of w for v overlaps in detector
//                                      units and in rows
// and G the sizes nx, ny, nz, nu, nv, na, spacings d, du, dv, offsets su, sv
// and out_scale.
//
// The one-thread-per-output kernels evaluate every weight, v overlaps
// included, for each (bin, voxel) pair: about 200 VALU instructions a pixel
// and bin.  Here a weight is evaluated once per (line, bin) or (view, column)
// by one lane and read by the wave, and lanes run along v (z): forward, a
// pixel's slabs are summed once for each of its rows and the bins' sums are
// matrix products; backward, a bin costs its rows' sum and one multiply-add.
// All sums are held in float64.  Measured, forward / backward: distance driven
// 128^3, 180 views of 192^2: 5.5 -> 0.82 ms / 2.7 -> 0.59 ms; separable footprint
// 120 x 132 x 101, 150 views of 187 x 150: 8.3 -> 0.98 ms / 2.1 -> 0.55 ms.
#pragma once
#include <algorithm>
#include <type_traits>

#include "vir_common.h"

namespace vir {

constexpr int kCtBins = 16;   // bins of a forward tile, accumulated in registers
constexpr int kCtWaves = 4;   // waves of a forward block: they share a tile's lines
constexpr int kCtLines = 4;   // lines whose lists a wave builds at once (16 bins x 4 lines = 64 lanes)
constexpr int kCtPix = 20;    // pixels of a line whose row sums are staged at once
constexpr int kCtList = 8;    // pixels of a line one bin's list holds
constexpr int kCtPitch = 68;  // of the row sums in LDS: 16-byte reads of four pixels' rows meet different banks
constexpr int kCtFoot = 6;    // bins a column's footprint list holds

__device__ __forceinline__ int ct_uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float ct_lane(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// First of the NS cells, of n >= NS, that an interval of at most NS - 1.01 cells
// (the launch checks that) from cell coordinate a on can meet: an interval of
// length L meets at most floor(L) + 2 cells.  a may be rounded.
template <int NS>
__device__ __forceinline__ float ct_first(float a, int n) {
    return fminf(fmaxf(floorf(a - (1e-3f + 4e-7f * (float)n)), 0.0f), (float)(n - NS));
}

// Overlaps w[0 .. NS-1] of [a, b] with the unit cells first, first + 1, ... of
// n cells whose edges lie at k - n/2.
template <int NS>
__device__ __forceinline__ int ct_cells(float a, float b, int n, double (&w)[NS]) {
    const float half = 0.5f * (float)n, f = ct_first<NS>(a + half, n);
    float e = f - half;
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const float e1 = e + 1.0f;
        w[q] = (double)fmaxf(fminf(e1, b) - fmaxf(e, a), 0.0f);
        e = e1;
    }
    return (int)f;
}

// The same of the detector interval [a, b] and cells of height h = 1/r on the
// detector, with edges at h (k - n/2): neighbouring cells share the rounded
// edge between them, so that the overlaps of an interval add up to its length.
template <int NS>
__device__ __forceinline__ int ct_slabs(float a, float b, float h, float r, int n, double (&w)[NS]) {
    const float half = 0.5f * (float)n, f = ct_first<NS>(__builtin_fmaf(a, r, half), n), k = f - half;
    float e = h * k;
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const float e1 = h * (k + (float)(q + 1));
        w[q] = (double)fmaxf(fminf(e1, b) - fmaxf(e, a), 0.0f);
        e = e1;
    }
    return (int)f;
}

// Weighted sum of NS consecutive values, in float64.
template <int NS>
__device__ __forceinline__ double ct_sum(const float* __restrict__ p, const double (&w)[NS]) {
    float x[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) x[q] = p[q];
    double s = (double)x[0] * w[0];
#pragma unroll
    for (int q = 1; q < NS; ++q) s = __builtin_fma((double)x[q], w[q], s);
    return s;
}

// The same where values of zero weight may be infinite: they do not count.
template <int NS>
__device__ __forceinline__ double ct_sum_some(const float* __restrict__ p, const double (&w)[NS]) {
    float x[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) x[q] = p[q];
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < NS; ++q) s = __builtin_fma((double)(w[q] > 0.0 ? x[q] : 0.0f), w[q], s);
    return s;
}

// ---------------------------------------------------------------- forward
//
// A block computes 16 bins x 64 rows of one view; its waves take groups of
// four lines in turn and add their float64 sums in wave order at the end, so
// the line loop has no barrier.  Per group a lane lists one (line, bin)'s
// pixels; per line the wave sums each pixel's slabs for its 64 rows into LDS
// (lane = row; consecutive lanes read consecutive z) and multiplies weights
// and sums on the matrix cores: v_mfma_f64_4x4x4_4b_f64, one block for each
// group of four bins with the pixels that group meets, four a step (two or
// three steps for pixels about as wide as bins, two fifths of the products of
// non-zero weight).  The row sums lie in LDS in float64, which leaves room for
// 20 pixels a wave with three blocks a CU; 16, 18 or 19 (pitch 72) and 24 (two
// blocks) are slower: distance driven, 128^3, 180 views of 192^2: 909, 881, 867,
// 1056 us against 821; separable footprint, 120 x 132 x 101, 150 views of 187 x
// 150: 1083, 1037, 1013, 1135 against 981.  (Sums in float32: 702 and 1099, with
// an error against float64 1.6 and 1.09 times as large.)  What bounds it: vector
// issue, most of it in the rows' slab sums and, with footprints, the weights.
struct CtWaveLds {
    double P[kCtPix * kCtPitch];
    float w[kCtLines * kCtBins * kCtList];
};

// One bin and row, pixel by pixel.
template <class M, class Geo, int NS>
__device__ double ct_fp_one(const Geo& G, const M& V, const float* __restrict__ vol, int iu, int iv) {
    const float vl = G.dv * (((float)iv - 0.5f * (float)G.nv) + G.sv);
    const float vr = G.dv * (((float)(iv + 1) - 0.5f * (float)G.nv) + G.sv);
    const float ul = G.du * (((float)iu - 0.5f * (float)G.nu) + G.su);
    const float ur = G.du * (((float)(iu + 1) - 0.5f * (float)G.nu) + G.su);
    const float fu = M::fp_unit(G);
    double acc = 0.0;
    for (int io = 0; io < V.no; ++io) {
        int k0 = 0, k1 = -1;
        if (!V.range(ul, ur, io, k0, k1)) continue;
        for (int k = k0; k <= k1; ++k) {
            const float w = V.weight(k, io, ul, ur);
            if (!(w > 0.0f)) continue;
            const float h = V.zmag(M::kLineMag ? 0 : k, io) * G.d;
            double ws[NS];
            const int z0 = ct_slabs<NS>(vl, vr, h, 1.0f / h, G.nz, ws);
            const int ix = V.xd ? k : io, iy = V.xd ? io : k;
            acc = __builtin_fma((double)(w * fu), ct_sum_some<NS>(vol + ((int64_t)ix * G.ny + iy) * G.nz + z0, ws), acc);
        }
    }
    return acc;
}

template <class M, class Geo, int NS>
__global__ __launch_bounds__(64 * kCtWaves) __attribute__((amdgpu_waves_per_eu(3))) void k_cone_fp_tile(Geo G, const float* __restrict__ ang,
                                                               const float* __restrict__ cs,
                                                               const float* __restrict__ sn,
                                                               const float* __restrict__ vol,
                                                               float* __restrict__ sino, int accumulate, int nut,
                                                               int nvt) {
    __shared__ __attribute__((aligned(16))) union {
        CtWaveLds wave[kCtWaves];
        double red[kCtWaves][kCtBins * 64];
    } lds;
    const int lane = threadIdx.x & 63;
    const int wave = ct_uni(threadIdx.x >> 6);
    CtWaveLds& L = lds.wave[wave];
    // operand slots: group (matrix block) mid; weights: bin lo, pixel hi; sums:
    // pixel hi, row quad lo; results: bin hi, row quad lo
    const int lo = lane & 3, mid = (lane >> 2) & 3, hi = lane >> 4;
    // place of row lane's sum: rows 16 c + 4 lo + e at 8 (2 c + e / 2) + 2 lo + e % 2,
    // so that the four row quads of a 16-byte read lie side by side
    const int slot = 8 * (2 * hi + (lo >> 1)) + 2 * mid + (lo & 1);
    int blk = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int v_lo = (blk % nvt) * 64;
    blk /= nvt;
    const int u_lo = (blk % nut) * kCtBins;
    blk /= nut;
    const int ia = blk % G.na;
    vol += (int64_t)(blk / G.na) * G.nx * G.ny * G.nz;            // batch item
    sino += (int64_t)(blk / G.na) * G.na * G.nu * G.nv;
    const M V(G, cs[ia], sn[ia], ang ? ang[ia] : 0.0f);
    // this lane's row, and the bin it lists pixels for
    const int iv = v_lo + lane;
    const float vl = G.dv * (((float)iv - 0.5f * (float)G.nv) + G.sv);
    const float vr = G.dv * (((float)(iv + 1) - 0.5f * (float)G.nv) + G.sv);
    const int iul = u_lo + (lane & 15);
    const float ul = G.du * (((float)iul - 0.5f * (float)G.nu) + G.su);
    const float ur = G.du * (((float)(iul + 1) - 0.5f * (float)G.nu) + G.su);
    const float fu = M::fp_unit(G);
    const int64_t kstride = (int64_t)(V.xd ? G.ny : 1) * G.nz, lstride = (int64_t)(V.xd ? 1 : G.ny) * G.nz;
    double acc[kCtBins];  // bin 4 mid + hi, rows 16 c + 4 lo + e at 4 c + e
#pragma unroll
    for (int i = 0; i < kCtBins; ++i) acc[i] = 0.0;

    for (int g = wave * kCtLines; g < V.no; g += kCtWaves * kCtLines) {
        int kf = 0, cnt = 0, k1 = -1;
        {
            const int io = g + (lane >> 4);
            int k0 = 0;
            if (io < V.no && iul < G.nu && !V.range(ul, ur, io, k0, k1)) k1 = -1;
            if (!(io < V.no && iul < G.nu)) k1 = -1;
            for (int k = k0; k <= k1; ++k) {
                const float w = V.weight(k, io, ul, ur);
                if (!(w > 0.0f)) {
                    if (cnt) break;  // the pixels of a bin are consecutive
                    continue;
                }
                if (!cnt) kf = k;
                if (cnt < kCtList) L.w[lane * kCtList + cnt] = w * fu;
                ++cnt;
            }
        }
        // more pixels a bin than a list holds (bins much wider than pixels):
        // the line is done in chunks of that many, each listed anew
        const bool over = __any(cnt > kCtList);
        // the pixels of a group of bins and of the line, and the line's steps
        int b0 = cnt ? kf : 0x7fffffff, b1 = cnt ? kf + cnt - 1 : -1;
#pragma unroll
        for (int m = 2; m >= 1; m >>= 1) {
            b0 = min(b0, __shfl_xor(b0, m));
            b1 = max(b1, __shfl_xor(b1, m));
        }
        const int gb = b1 >= 0 ? b0 : 0;
        int steps = b1 >= 0 ? (b1 - b0 + 4) >> 2 : 0;
#pragma unroll
        for (int m = 8; m >= 4; m >>= 1) {
            b0 = min(b0, __shfl_xor(b0, m));
            b1 = max(b1, __shfl_xor(b1, m));
            steps = max(steps, __shfl_xor(steps, m));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a wave's LDS accesses are in order
        for (int l = 0; l < kCtLines && g + l < V.no; ++l) {
            const int io = g + l;
            const int kb = __builtin_amdgcn_readlane(b0, 16 * l), ke = __builtin_amdgcn_readlane(b1, 16 * l);
            if (ke < 0) continue;
            const int nks = __builtin_amdgcn_readlane(steps, 16 * l);
            // this operand slot's list
            const int e = 16 * l + (lane & 15);
            const int kfe = __shfl(kf, e), cne = __shfl(cnt, e), win = __shfl(gb, e) + hi;
            double ws[NS];
            int z0 = 0;
            if (M::kLineMag) {
                const float h = V.zmag(0, io) * G.d;
                z0 = ct_slabs<NS>(vl, vr, h, 1.0f / h, G.nz, ws);
            }
            const int step = over ? kCtList : kCtPix;
            for (int kc = kb; kc <= ke; kc += step) {
                const int nk = min(step, ke - kc + 1);
                if (over && (lane >> 4) == l)
                    for (int k = max(kf, kc); k < min(kf + cnt, kc + nk); ++k)
                        L.w[lane * kCtList + k - kc] = V.weight(k, io, ul, ur) * fu;
                float hk = 0.0f, rk = 0.0f;  // lane = pixel
                if (!M::kLineMag) {
                    hk = V.zmag(min(kc + lane, V.nd - 1), io) * G.d;
                    rk = 1.0f / hk;
                }
                const float* col = vol + (int64_t)io * lstride + (int64_t)kc * kstride;
                auto stage = [&](int kk, const float* p) {
                    if (!M::kLineMag) z0 = ct_slabs<NS>(vl, vr, ct_lane(hk, kk), ct_lane(rk, kk), G.nz, ws);
                    return ct_sum<NS>(p + z0, ws);
                };
                int kk = 0;
                for (; kk + 3 < nk; kk += 4, col += 4 * kstride) {
                    double p[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) p[t] = stage(kk + t, col + t * kstride);
#pragma unroll
                    for (int t = 0; t < 4; ++t) L.P[(kk + t) * kCtPitch + slot] = p[t];
                }
                for (; kk < nk; ++kk, col += kstride) L.P[kk * kCtPitch + slot] = stage(kk, col);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const int k0 = over ? kc + hi : win, ns = over ? (nk + 3) >> 2 : nks, wb = over ? kc : kfe;
                for (int t = 0; t < ns; ++t) {
                    const int k = k0 + 4 * t, kr = k - kc;
                    const bool in = (unsigned)(k - kfe) < (unsigned)cne && (unsigned)kr < (unsigned)nk;
                    if (!__any(in)) continue;  // another chunk's pixels
                    const double w = in ? (double)L.w[e * kCtList + (k - wb)] : 0.0;
                    const double2* row = (const double2*)(L.P + min(max(kr, 0), nk - 1) * kCtPitch + 2 * lo);
                    double2 x[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c) x[c] = row[4 * c];
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        acc[2 * c] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, x[c].x, acc[2 * c], 0, 0, 0);
                        acc[2 * c + 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, x[c].y, acc[2 * c + 1], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kCtBins; ++i) lds.red[wave][i * 64 + lane] = acc[i];
    __syncthreads();
    if (iv >= G.nv) return;
    for (int i = wave; i < kCtBins; i += kCtWaves) {
        const int iu = u_lo + i;
        if (iu >= G.nu) break;
        // bin i, row lane: sum 4 (lane / 16) + lane % 4 of slot mid = i / 4, hi = i % 4
        const int e = (4 * (lane >> 4) + lo) * 64 + 16 * (i & 3) + 4 * (i >> 2) + mid;
        double s = lds.red[0][e];
#pragma unroll
        for (int w = 1; w < kCtWaves; ++w) s += lds.red[w][e];
        if (!(fabs(s) < (double)VIR_INF)) s = ct_fp_one<M, Geo, NS>(G, V, vol, iu, iv);  // zero weights times infinities
        const int64_t o = ((int64_t)ia * G.nu + iu) * G.nv + iv;
        float r = (float)s * G.out_scale;
        if (accumulate) r += sino[o];
        sino[o] = r;
    }
}

// --------------------------------------------------------------- backward
//
// A wave owns a column of 64 voxels (lane = z).  For 64 views at a time, lane
// = view lists the bins that the column's pixel meets; the view loop then
// reads the list by readlane and each lane sums the NS rows its slab meets
// of every bin.
//
// Zero weights times infinite values make NaNs: a sum that is not finite is
// formed again without them.

// Bins [j0, j1] that pixel k of line io can meet in view V.
template <class M, class Geo>
__device__ __forceinline__ void ct_bins(const Geo& G, const M& V, int k, int io, int& j0, int& j1) {
    const float inv_du = 1.0f / G.du, u0 = G.du * (-0.5f * (float)G.nu + G.su);
    const float mar = 0.01f + 1e-6f * (float)G.nu;  // rounding of the bin positions
    float lo, hi;
    V.foot(k, io, lo, hi);
    j0 = (int)fmaxf(floorf((lo - u0) * inv_du - mar), 0.0f);
    j1 = (int)fminf(floorf((hi - u0) * inv_du + mar), (float)(G.nu - 1));
}

// One voxel, bin by bin.
template <class M, class Geo, int NS>
__device__ double ct_bp_one(const Geo& G, const float* __restrict__ ang, const float* __restrict__ cs,
                            const float* __restrict__ sn, const float* __restrict__ sino, int ix, int iy, int iz) {
    const auto edge = [&](int j) { return G.du * (((float)j - 0.5f * (float)G.nu) + G.su); };
    const float zl = G.d * ((float)iz - 0.5f * (float)G.nz), zr = G.d * ((float)(iz + 1) - 0.5f * (float)G.nz);
    double acc = 0.0;
    for (int ia = 0; ia < G.na; ++ia) {
        const M V(G, cs[ia], sn[ia], ang ? ang[ia] : 0.0f);
        const int k = V.xd ? ix : iy, io = V.xd ? iy : ix;
        int j0, j1;
        ct_bins(G, V, k, io, j0, j1);
        const float m = V.zmag(k, io) / G.dv;
        double ws[NS];
        const int m0 = ct_cells<NS>(__builtin_fmaf(zl, m, -G.sv), __builtin_fmaf(zr, m, -G.sv), G.nv, ws);
        for (int j = j0; j <= j1; ++j) {
            const float w = V.weight(k, io, edge(j), edge(j + 1));
            if (w > 0.0f)
                acc = __builtin_fma((double)w, ct_sum_some<NS>(sino + ((int64_t)ia * G.nu + j) * G.nv + m0, ws), acc);
        }
    }
    return acc;
}

template <class M, class Geo, int NS>
__global__ __launch_bounds__(256) void k_cone_bp_col(Geo G, const float* __restrict__ ang,
                                                    const float* __restrict__ cs, const float* __restrict__ sn,
                                                    const float* __restrict__ sino, float* __restrict__ vol,
                                                    int accumulate, int nzt, int64_t ncol) {
    const int lane = threadIdx.x & 63;
    const int64_t wid = xcd_remap(blockIdx.x, gridDim.x) * 4 + ct_uni(threadIdx.x >> 6);
    if (wid >= ncol) return;  // whole wave
    const int iz = (int)(wid % nzt) * 64 + lane;
    int64_t r = wid / nzt;
    const int iy = (int)(r % G.ny);
    r /= G.ny;
    const int ix = (int)(r % G.nx);
    vol += (r / G.nx) * G.nx * G.ny * G.nz;
    sino += (r / G.nx) * (int64_t)G.na * G.nu * G.nv;
    const float zl = G.d * ((float)iz - 0.5f * (float)G.nz), zr = G.d * ((float)(iz + 1) - 0.5f * (float)G.nz);
    double acc = 0.0;
    for (int va = 0; va < G.na; va += 64) {
        int cnt = 0, jf = 0;
        float w[kCtFoot], zs = 0.0f;
#pragma unroll
        for (int t = 0; t < kCtFoot; ++t) w[t] = 0.0f;
        const int ial = min(va + lane, G.na - 1);
        const M V(G, cs[ial], sn[ial], ang ? ang[ial] : 0.0f);
        const int k = V.xd ? ix : iy, io = V.xd ? iy : ix;
        int j0, j1;
        ct_bins(G, V, k, io, j0, j1);
        const auto edge = [&](int j) { return G.du * (((float)j - 0.5f * (float)G.nu) + G.su); };
        for (int j = j0; j <= j1; ++j) {
            const float x = V.weight(k, io, edge(j), edge(j + 1));
            if (!(x > 0.0f)) {
                if (cnt) break;
                continue;
            }
            if (!cnt) jf = j;
#pragma unroll
            for (int t = 0; t < kCtFoot; ++t) w[t] = t == cnt ? x : w[t];
            ++cnt;
        }
        zs = V.zmag(k, io) / G.dv;
        const bool over = __any(cnt > kCtFoot);  // bins much finer than pixels
        const int nvw = min(64, G.na - va);
        for (int v = 0; v < nvw; ++v) {
            const int n = __builtin_amdgcn_readlane(cnt, v);
            if (n == 0) continue;
            const int j = __builtin_amdgcn_readlane(jf, v);
            const float m = ct_lane(zs, v);
            double ws[NS];
            const int m0 = ct_cells<NS>(__builtin_fmaf(zl, m, -G.sv), __builtin_fmaf(zr, m, -G.sv), G.nv, ws);
            const float* row = sino + ((int64_t)(va + v) * G.nu + j) * G.nv + m0;
            if (over) {
                const M W(G, cs[va + v], sn[va + v], ang ? ang[va + v] : 0.0f);
                const int kv = W.xd ? ix : iy, iov = W.xd ? iy : ix;
                for (int t = 0; t < n; ++t)
                    acc = __builtin_fma((double)W.weight(kv, iov, edge(j + t), edge(j + t + 1)),
                                        ct_sum<NS>(row + (int64_t)t * G.nv, ws), acc);
                continue;
            }
            if (n >= 2) {
                const double s0 = ct_sum<NS>(row, ws), s1 = ct_sum<NS>(row + G.nv, ws);
                acc = __builtin_fma((double)ct_lane(w[0], v), s0, acc);
                acc = __builtin_fma((double)ct_lane(w[1], v), s1, acc);
            } else {
                acc = __builtin_fma((double)ct_lane(w[0], v), ct_sum<NS>(row, ws), acc);
            }
#pragma unroll
            for (int t = 2; t < kCtFoot; ++t) {
                if (t >= n) break;
                acc = __builtin_fma((double)ct_lane(w[t], v), ct_sum<NS>(row + (int64_t)t * G.nv, ws), acc);
            }
        }
    }
    if (iz >= G.nz) return;
    if (!(fabs(acc) < (double)VIR_INF)) acc = ct_bp_one<M, Geo, NS>(G, ang, cs, sn, sino, ix, iy, iz);
    const int64_t o = ((int64_t)ix * G.ny + iy) * G.nz + iz;
    float res = (float)(acc * (double)M::bp_unit(G)) * G.out_scale;
    if (accumulate) res += vol[o];
    vol[o] = res;
}

// One thread per voxel, with the column kernel's terms in its order: the same bits.
template <class M, class Geo, int NS>
__global__ __launch_bounds__(256) void k_cone_bp_vox(Geo G, const float* __restrict__ ang,
                                                    const float* __restrict__ cs, const float* __restrict__ sn,
                                                    const float* __restrict__ sino, float* __restrict__ vol,
                                                    int accumulate, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    int64_t r = t / G.nz;
    const int iz = (int)(t % G.nz), iy = (int)(r % G.ny);
    r /= G.ny;
    const int ix = (int)(r % G.nx);
    sino += (r / G.nx) * (int64_t)G.na * G.nu * G.nv;
    const double acc = ct_bp_one<M, Geo, NS>(G, ang, cs, sn, sino, ix, iy, iz);
    float res = (float)(acc * (double)M::bp_unit(G)) * G.out_scale;
    if (accumulate) res += vol[t];
    vol[t] = res;
}

// Cells a v (z) interval of at most `len` cells can meet, as the NS of the
// kernels above, or 0 where they do not apply (intervals longer than 2.9
// cells, fewer than NS cells in all, or so many that ct_first's margin would
// not fit).
inline int ct_slots(double len, int n) {
    const int ns = len <= 0.99 ? 2 : len <= 1.99 ? 3 : len <= 2.9 ? 4 : 0;
    return n >= ns && n <= 20000 ? ns : 0;
}

// True when the forward tile, whose 64 lanes run along v, is slower than one
// thread per output: up to four rows, and blocks of one item (so that its bits
// don't depend on the batch) that fill the chip several times over.  Tile | per
// output, us, rows as slabs, distance driven: 256^2, 360 views (8640 blocks) 3 rows
// 1701 | 1305, 4: 1709 | 1522, 6: (32 slabs) 2041 | 2204; 128^2, 360 views (4320)
// 3: 508 | 441, 4: 500 | 538; 256^2, 60 views (1440) 3: 371 | 630; 181 x 94 x 2, 306
// views of 123 x 3 (2448) 537 | 466.
template <class Geo>
bool ct_few_rows(const Geo& G) {
    return G.nv <= 4 && (int64_t)G.na * ((G.nu + kCtBins - 1) / kCtBins) > (G.nv < 4 ? 2300 : 4400);
}

// Threads that one item's launch takes.
template <class Geo>
int64_t ct_threads(const Geo& G, bool fp) {
    return fp ? (int64_t)G.na * ((G.nu + kCtBins - 1) / kCtBins) * ((G.nv + 63) / 64) * 256
              : (int64_t)G.nx * G.ny * ((G.nz + 63) / 64) * 64 + 256;
}

template <class M, class Geo>
int ct_fp(const Geo& G, int nb, int ns, const float* ang, const float* cosv, const float* sinv, const float* vol,
          float* sino, int acc, hipStream_t st, const char* what) {
    const int nut = (G.nu + kCtBins - 1) / kCtBins, nvt = (G.nv + 63) / 64;
    const dim3 grd((unsigned)((int64_t)nb * G.na * nut * nvt)), blk(64 * kCtWaves);
    if (ns == 2)
        hipLaunchKernelGGL((k_cone_fp_tile<M, Geo, 2>), grd, blk, 0, st, G, ang, cosv, sinv, vol, sino, acc, nut, nvt);
    else if (ns == 3)
        hipLaunchKernelGGL((k_cone_fp_tile<M, Geo, 3>), grd, blk, 0, st, G, ang, cosv, sinv, vol, sino, acc, nut, nvt);
    else
        hipLaunchKernelGGL((k_cone_fp_tile<M, Geo, 4>), grd, blk, 0, st, G, ang, cosv, sinv, vol, sino, acc, nut, nvt);
    return check_hip(hipGetLastError(), what);
}

template <class M, class Geo>
int ct_bp(const Geo& G, int nb, int ns, const float* ang, const float* cosv, const float* sinv, const float* sino,
          float* vol, int acc, hipStream_t st, const char* what) {
    const int nzt = (G.nz + 63) / 64;
    const int64_t ncol = (int64_t)nb * G.nx * G.ny * nzt;
    // Thin volumes leave most lanes of a column idle: with more columns than fill
    // the chip a thread a voxel is faster up to about 18 slabs, and with few
    // views, for which a column's lists cost as much as for 64, up to more.  A
    // thousand columns take about 0.42 us every 64 views and 0.09 a view; a view
    // 0.4 us and 0.33 a thousand waves of voxels.  Columns | voxels in us, distance driven, 60 views: 64^2 x 8 38 | 54;
    // 128^2 x 4 106 | 55, x 12 105 | 83, x 16 105 | 101; 256^2 x 3 371 | 82, x 8 368 |
    // 178, x 16 371 | 332; 512^2 x 16, 30 views, 772 | 638, x 70 1558 | 2708.  Both give
    // the same bits, so the batch may count.
    const int64_t n = (int64_t)nb * G.nx * G.ny * G.nz;
    const bool thin = (double)G.nz / nzt < 17.5 + 82.0 * ((G.na + 63) / 64) / std::max(G.na, 1) - 7.8e4 / (double)ncol;
    const dim3 grd((unsigned)(((thin ? (n + 63) / 64 : ncol) + 3) / 4)), blk(256);
    const auto run = [&](auto slots) {
        constexpr int NS = decltype(slots)::value;
        if (thin)
            hipLaunchKernelGGL((k_cone_bp_vox<M, Geo, NS>), grd, blk, 0, st, G, ang, cosv, sinv, sino, vol, acc, n);
        else
            hipLaunchKernelGGL((k_cone_bp_col<M, Geo, NS>), grd, blk, 0, st, G, ang, cosv, sinv, sino, vol, acc, nzt, ncol);
    };
    if (ns == 2) run(std::integral_constant<int, 2>{});
    else if (ns == 3) run(std::integral_constant<int, 3>{});
    else run(std::integral_constant<int, 4>{});
    return check_hip(hipGetLastError(), what);
}

}  // namespace vir
