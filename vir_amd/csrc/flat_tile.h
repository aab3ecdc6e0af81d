// 2-D footprint projections in tiles, shared by the distance-driven (dd.hip)
// and separable-footprint (sf.hip) projectors.
//
// In both models a pixel casts an interval on the detector, with a factor,
// and weighs a bin by factor * overlap.  A model M gives, per view:
//   M(G, v)                 the view, from its trigonometry (M::Trig)
//   xd, nd, no              driving axis, pixels a line, lines
//   centre(io)              orthogonal coordinate of line io
//   lin(u, A, B)            detector coordinate u inverted along a line with
//                           coordinate oc: pixel position A - oc B; returns
//                           the denominator, zero for rays along the line
//   margin()                largest distance of a pixel's interval end from
//                           the position lin() inverts (kCentre models: of
//                           its centre; others invert pixel edges, margin 0)
//   line_factor(oc)         the factor's part that a line shares (forward)
//   edge(k, oc)             lower edge of pixel k (kShared models: pixels of a
//                           line share their edges)
//   pixel(k, io, u0, u1)    interval of pixel k, returns its own factor (the
//                           other models)
//   bp_unit(G)              factor of the quad's factors (backward)
//   grid(k, io), amp(k, io) its interval spans the corners grid() of its two
//                           ends and edges, its factor is amp() (kCorners)
//   quad(ix, iy, ...)       intervals and factors of a 2 x 2 pixel block
//
// The one-thread-per-output kernels repeat the interval of a pixel for every
// bin that tries it, or its trigonometry for every pixel.  Here an interval is
// evaluated once per line and tile (forward) or shared by a 2 x 2 block
// (backward), and no wave waits for another until the sums are added: the
// waves of a block share the lines (views) of a tile and add their float64
// sums in wave order.  Measured, forward / backward: distance-driven fan 512^2,
// 720 views of 888 bins: 1.88 -> 0.85 ms / 1.18 -> 0.64 ms (the forward was a
// tile of 256 bins with two barriers a line pair and waited in 62 % of its
// cycles); separable-footprint fan 256^2, 360 views of 444: 2.01 -> 0.37 ms /
// 0.43 -> 0.10 ms.  VALU work bounds both directions.
#pragma once
#include "vir_common.h"

namespace vir {

__device__ __forceinline__ int ft_uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float ft_lane(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// Sum of all chains, of which wave w of NW has added its own (w, w + NW, ..) up:
// in the order of four waves.
template <int NW, class Part>
__device__ __forceinline__ double ft_chains(Part&& part) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        double t = part(w);
#pragma unroll
        for (int c = w + 4; c < NW; c += 4) t += part(c);
        s = w == 0 ? t : s + t;
    }
    return s;
}

constexpr int kFtBins = 128;   // bins of a forward tile, two a lane
constexpr int kFtStage = 128;  // interval slots of a line staged at once
constexpr int kFtPad = 6;      // of which empty ones past the last pixel, read but of no overlap

// ---------------------------------------------------------------- forward
//
// A bin's lines are summed in kFtLines chains (line modulo kFtLines) and the
// chains in one order, whatever the number of waves, so that an item's bits do
// not depend on the batch it is in (at most 2 % of the time).
constexpr int kFtLines = 8;

template <bool SHARED>
struct FtWaveLds {  // an edge and a value per pixel
    float e[2][kFtStage + 2];
    float v[2][kFtStage];
};
template <>
struct FtWaveLds<false> {  // interval, value, factor
    float4 p[2][kFtStage];
};

template <class M, class Geo, int NW>
__global__ __launch_bounds__(64 * NW) void k_fp2d_tile(Geo G, const float* __restrict__ ang,
                                                      const float* __restrict__ cs, const float* __restrict__ sn,
                                                      const float* __restrict__ img, float* __restrict__ sino,
                                                      int accumulate, int nut, SirtEpi E) {
    __shared__ union {
        FtWaveLds<M::kShared> wave[NW];
        double red[NW][kFtBins];
    } lds;
    const int lane = threadIdx.x & 63;
    const int wave = ft_uni(threadIdx.x >> 6);
    auto& L = lds.wave[wave];
    const int u_lo = (blockIdx.x % nut) * kFtBins;
    const int64_t row = blockIdx.x / nut;  // batch item and view
    const int ia = (int)(row % G.na);
    img += (row / G.na) * G.nx * G.ny;
    const M V(G, typename M::Trig(cs[ia], sn[ia], ang ? ang[ia] : 0.0f));
    // (a view without a finite angle meets nothing)
    const int nd = V.nd, no = fabsf(cs[ia]) + fabsf(sn[ia]) < VIR_INF ? V.no : 0;
    const float half = 0.5f * (float)nd, inv_d = 1.0f / G.d;
    const auto edge = [&](int j) { return G.du * (((float)j - 0.5f * (float)G.nu) + G.su); };
    // pixel range of the interval [u0, u1]: position p0 - oc q0 .. p1 - oc q1,
    // widened by eps for the rounding of a position (a sum of such terms).  An
    // interval with a ray along the line inside, where positions run through
    // infinity, takes the whole line.
    struct Inv { float p0, q0, p1, q1, eps; };
    const auto invert = [&](float u0, float u1) {
        Inv r;
        const float e0 = V.lin(u0 - V.margin(), r.p0, r.q0), e1 = V.lin(u1 + V.margin(), r.p1, r.q1);
        if (!(e0 * e1 > 1e-6f)) return Inv{-1e9f, 0.0f, 1e9f, 0.0f, 0.0f};
        const float c = M::kCentre ? half - 0.5f : half;
        r.p0 = __builtin_fmaf(r.p0, inv_d, c);
        r.p1 = __builtin_fmaf(r.p1, inv_d, c);
        r.q0 *= inv_d;
        r.q1 *= inv_d;
        r.eps = 2e-3f + 2e-6f * (float)(nd + no) +
                4e-7f * (fmaxf(fabsf(r.p0), fabsf(r.p1)) + 0.5f * (float)no * fmaxf(fabsf(r.q0), fabsf(r.q1)));
        return r;
    };
    const auto range = [&](const Inv& r, float oc, float& a, float& b) {
        const float x0 = __builtin_fmaf(-oc, r.q0, r.p0), x1 = __builtin_fmaf(-oc, r.q1, r.p1);
        a = fminf(x0, x1) - r.eps;
        b = floorf(fmaxf(x0, x1) + r.eps);
        a = M::kCentre ? ceilf(a) : floorf(a);
    };
    float ul[2], ur[2];
    Inv I[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int iu = u_lo + 64 * q + lane;
        ul[q] = edge(iu);
        ur[q] = edge(iu + 1);
        I[q] = invert(ul[q], ur[q]);
    }
    const Inv T = invert(edge(u_lo), edge(min(u_lo + kFtBins, G.nu)));
    double acc[2], sum[2] = {0.0, 0.0};
    // this bin's pixels of line slot h, pixels kc .. kc + nk - 1 staged
    const auto merge = [&](int h, float oc, float lf, int kc, int nk) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float a, b;
            range(I[q], oc, a, b);
            const int k0 = (int)fmaxf(a, (float)kc) - kc, k1 = (int)fminf(b, (float)(kc + nk - 1)) - kc;
            if (k1 < k0) continue;
            const auto term = [&](int k) {
                float x, y, v, w = lf;
                if constexpr (M::kShared) {
                    x = L.e[h][k];
                    y = L.e[h][k + 1];
                    v = L.v[h][k];
                } else {
                    const float4 p = L.p[h][k];
                    x = p.x;
                    y = p.y;
                    v = p.z;
                    w = p.w;
                }
                const float ov = fminf(fmaxf(x, y), ur[q]) - fmaxf(fminf(x, y), ul[q]);
                w = M::kShared ? ov * lf : (ov * lf) * w;
                w = v * w;
                acc[q] += (double)(ov > 0.0f ? w : 0.0f);
            };
#pragma unroll
            for (int t = 0; t < M::kFixed; ++t) term(k0 + t);  // past k1: no overlap, or an empty slot
            for (int k = k0 + M::kFixed; k <= k1; ++k) term(k);
        }
    };
    const int stride = V.xd ? G.ny : 1, lstride = V.xd ? 1 : G.ny;
    constexpr int STEP = kFtLines / NW;  // chains of a wave: wave, wave + NW, ..
    for (int ch = 0; ch < STEP; ++ch) {
        acc[0] = acc[1] = 0.0;
        for (int g = 0; g < no; g += 64 * NW) {
            // lane = line g + NW lane + wave: its coordinate, pixel band and factor
            const int iol = g + NW * lane + wave;
            const float ocl = V.centre(min(iol, no - 1));
            const float lfl = V.line_factor(ocl);
            float a, b;
            range(T, ocl, a, b);
            const int kbl = (int)fmaxf(a - 1.0f, 0.0f);
            const int kel = iol < no ? (int)fminf(b + 1.0f, (float)(nd - 1)) : -1;
            const int nl = min(64, (no - g - wave + NW - 1) / NW);
            for (int l = ch; l < nl; l += 2 * STEP) {
                int kb[2], ke[2];
                float oc[2], lf[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int t = min(l + STEP * h, 63);
                    kb[h] = __builtin_amdgcn_readlane(kbl, t);
                    ke[h] = l + STEP * h < nl ? __builtin_amdgcn_readlane(kel, t) : -1;
                    oc[h] = ft_lane(ocl, t);
                    lf[h] = ft_lane(lfl, t);
                }
                const int most = max(ke[0] - kb[0], ke[1] - kb[1]);
                for (int c = 0; c <= most; c += kFtStage - kFtPad) {
                    int kc[2], nk[2];
                    float x[2][2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        kc[h] = kb[h] + c;
                        nk[h] = min(kFtStage - kFtPad, ke[h] - kc[h] + 1);
                        const int io = g + NW * (l + STEP * h) + wave;
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const int k = 64 * t + lane;
                            x[h][t] = 0.0f;
                            if (k < nk[h]) x[h][t] = img[(int64_t)(kc[h] + k) * stride + (int64_t)io * lstride];
                        }
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int io = g + NW * (l + STEP * h) + wave;
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const int k = 64 * t + lane;
                            if (64 * t >= nk[h] + kFtPad) continue;  // whole wave
                            // slots past the last pixel are empty: both ends at
                            // one place
                            if constexpr (M::kShared) {
                                L.e[h][k] = V.edge(min(kc[h] + k, kc[h] + nk[h]), oc[h]);
                                L.v[h][k] = x[h][t];
                            } else if constexpr (!M::kCorners) {
                                float u0, u1;
                                const float f = V.pixel(min(kc[h] + k, nd - 1), min(io, no - 1), u0, u1);
                                L.p[h][k] = make_float4(u0, k < nk[h] ? u1 : u0, x[h][t], f);
                            }
                        }
                        if constexpr (M::kCorners) {
                            // the corners at pixel k's lower end, the line's two
                            // edges; the next lane's are those at its upper end
                            // (four divisions a pixel for six: 0.41 -> 0.39 ms)
                            const int il = min(io, no - 1);
                            if (nk[h] + kFtPad <= 0) continue;     // whole wave
                            const bool two = nk[h] + kFtPad > 64;  // whole wave
                            float lo[2], hi[2];
#pragma unroll
                            for (int t = 0; t < 2; ++t) {
                                lo[t] = hi[t] = 0.0f;
                                if (t && !two) continue;
                                const float c0 = V.grid(min(kc[h] + 64 * t + lane, nd), il);
                                const float c1 = V.grid(min(kc[h] + 64 * t + lane, nd), il + 1);
                                lo[t] = fminf(c0, c1);
                                hi[t] = fmaxf(c0, c1);
                            }
#pragma unroll
                            for (int t = 0; t < 2; ++t) {
                                if (t && !two) continue;
                                const int k = 64 * t + lane;
                                float ln = __shfl_down(lo[t], 1), hn = __shfl_down(hi[t], 1);
                                if (t == 0) {  // (slots 63, if there is no second half, and 127 are empty)
                                    ln = lane == 63 ? ft_lane(lo[1], 0) : ln;
                                    hn = lane == 63 ? ft_lane(hi[1], 0) : hn;
                                }
                                const float u0 = fminf(lo[t], ln), u1 = fmaxf(hi[t], hn);
                                L.p[h][k] = make_float4(u0, k < nk[h] ? u1 : u0, x[h][t],
                                                        V.amp(min(kc[h] + k, nd - 1), il));
                            }
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a wave's LDS accesses are in order
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        if (nk[h] > 0) merge(h, oc[h], lf[h], kc[h], nk[h]);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
            }
        }
        sum[0] += acc[0];
        sum[1] += acc[1];
    }
    __syncthreads();
    lds.red[wave][lane] = sum[0];
    lds.red[wave][64 + lane] = sum[1];
    __syncthreads();
    for (int i = threadIdx.x; i < kFtBins; i += 64 * NW) {
        const int iu = u_lo + i;
        if (iu >= G.nu) continue;
        const double s = ft_chains<NW>([&](int w) { return lds.red[w][i]; });
        const int64_t o = row * G.nu + iu;
        float r = (float)s * G.out_scale;
        if (accumulate) r += sino[o];
        sirt_store(E, sino, o, r);
    }
}

// --------------------------------------------------------------- backward
//
// A block takes 16 x 16 pixels, a 2 x 2 block a lane; wave w of its NW takes
// views w, w + NW, ..., in chains (view modulo kFtViews) as the forward's lines.
constexpr int kFtViews = 16;

template <class M, class Geo, int NW>
__global__ __launch_bounds__(64 * NW) void k_bp2d_tile(Geo G, const float* __restrict__ ang,
                                                      const float* __restrict__ cs, const float* __restrict__ sn,
                                                      const float* __restrict__ sino, float* __restrict__ img,
                                                      int accumulate, int nty, int nt, SirtEpi E) {
    __shared__ double red[NW][256];
    const int lane = threadIdx.x & 63;
    const int wave = ft_uni(threadIdx.x >> 6);
    const int tile = blockIdx.x % nt;
    const int64_t item = blockIdx.x / nt;
    sino += item * G.na * G.nu;
    const int bx = (tile / nty) * 16, by = (tile % nty) * 16;
    const int ix = bx + 2 * (lane >> 3), iy = by + 2 * (lane & 7);
    const float inv_du = 1.0f / G.du, half = 0.5f * (float)G.nu;
    // u in bins from the first one's edge, and its rounding
    const float off = half - G.su, mar = 1e-4f + 1e-6f * ((float)G.nu + fabsf(G.su));
    const float uend = G.du * (half + G.su);
    double acc[4], sum[4] = {0.0, 0.0, 0.0, 0.0};
    constexpr int STEP = kFtViews / NW;  // chains of a wave: wave, wave + NW, ..
    for (int ch = 0; ch < STEP; ++ch) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = 0.0;
        for (int g = 0; g < G.na; g += 64 * NW) {
            const int il = min(g + NW * lane + wave, G.na - 1);
            const typename M::Trig tl(cs[il], sn[il], ang ? ang[il] : 0.0f);  // lane = view
            // (a comparison with infinity inside the ballot is compiled to one that NaN passes)
            const uint64_t finite = __ballot(0.0f * cs[il] + 0.0f * sn[il] == 0.0f);
            const int nl = min(64, (G.na - g - wave + NW - 1) / NW);
            for (int l = ch; l < nl; l += STEP) {
                if (!((finite >> l) & 1)) continue;
                const M V(G, tl.lane(l));
                const float* __restrict__ row = sino + (int64_t)(g + NW * l + wave) * G.nu;
                float lo[4], hi[4], f[4];
                V.quad(ix, iy, lo, hi, f);
                int j0[4], n[4];
                float y[4][3];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    hi[q] = fminf(hi[q], uend);
                    const float j = fminf(fmaxf(floorf(__builtin_fmaf(lo[q], inv_du, off) - mar), 0.0f), (float)(G.nu - 1));
                    j0[q] = (int)j;
                    n[q] = (int)fminf(__builtin_fmaf(hi[q], inv_du, off) + mar, (float)(G.nu - 1)) - j0[q];  // bins past the first
#pragma unroll
                    for (int t = 0; t < 3; ++t) y[q][t] = row[min(j0[q] + t, G.nu - 1)];
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    double s = 0.0;
                    // neighbouring bins share the rounded edge between them, so a
                    // pixel's overlaps add up to its interval
                    float k = ((float)j0[q] - half) + G.su, e = G.du * k;
                    const auto term = [&](float v) {
                        k += 1.0f;
                        const float e1 = G.du * k, ov = fminf(hi[q], e1) - fmaxf(lo[q], e);
                        s += (double)(ov > 0.0f ? v * ov : 0.0f);
                        e = e1;
                    };
#pragma unroll
                    for (int t = 0; t < 3; ++t) term(y[q][t]);
                    for (int t = 3; t <= n[q]; ++t) term(row[j0[q] + t]);
                    acc[q] = __builtin_fma(s, (double)f[q], acc[q]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) sum[q] += acc[q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave][64 * q + lane] = sum[q];
    __syncthreads();
    const double unit = (double)M::bp_unit(G);
    for (int i = threadIdx.x; i < 256; i += 64 * NW) {
        // consecutive threads, consecutive pixels: px (i / 16, i % 16)
        const int x = i >> 4, y = i & 15;
        const int slot = 64 * (2 * (x & 1) + (y & 1)) + 8 * (x >> 1) + (y >> 1);
        if (bx + x >= G.nx || by + y >= G.ny) continue;
        const double s = ft_chains<NW>([&](int w) { return red[w][slot]; });
        const int64_t o = (item * G.nx + bx + x) * G.ny + by + y;
        float r = (float)(s * unit) * G.out_scale;
        if (accumulate) r += img[o];
        sirt_store(E, img, o, r);
    }
}

// Threads that one item's launch takes (at most; fewer where a batch has more tiles).
template <class Geo>
int64_t ft_threads(const Geo& G, bool fp) {
    const int64_t n = fp ? (int64_t)G.na * ((G.nu + kFtBins - 1) / kFtBins) : (int64_t)((G.nx + 15) / 16) * ((G.ny + 15) / 16);
    return n * (n >= 2048 ? 256 : fp ? 512 : 1024);
}

// Waves that share a tile: four, or sixteen (eight forward) where the tiles
// alone would leave CUs without work (forward: in less than about two rounds of
// resident waves, the edge tiles' short bands leave some idle; four | eight
// waves, footprint fan pair at 256^2, 360 views, 1440 tiles: 454 | 437 us,
// distance-driven arc pair with 2 iterations 557 | 541; 400^2, 1800: 819 | 799,
// 1043 | 1035; 600^2, 2880: no difference).
template <class M, class Geo>
int ft_fp(const Geo& G, int nb, const float* ang, const float* cosv, const float* sinv, const float* img,
          float* sino, int acc, hipStream_t st, const SirtEpi& E, const char* what) {
    const int nut = (G.nu + kFtBins - 1) / kFtBins;
    const int64_t n = (int64_t)nb * G.na * nut;
    if (n >= 2048)
        hipLaunchKernelGGL((k_fp2d_tile<M, Geo, 4>), dim3((unsigned)n), dim3(256), 0, st, G, ang, cosv, sinv, img,
                           sino, acc, nut, E);
    else
        hipLaunchKernelGGL((k_fp2d_tile<M, Geo, 8>), dim3((unsigned)n), dim3(512), 0, st, G, ang, cosv, sinv, img,
                           sino, acc, nut, E);
    return check_hip(hipGetLastError(), what);
}

template <class M, class Geo>
int ft_bp(const Geo& G, int nb, const float* ang, const float* cosv, const float* sinv, const float* sino,
          float* img, int acc, hipStream_t st, const SirtEpi& E, const char* what) {
    const int nty = (G.ny + 15) / 16, nt = ((G.nx + 15) / 16) * nty;
    const int64_t n = (int64_t)nb * nt;
    if (n >= 1024)
        hipLaunchKernelGGL((k_bp2d_tile<M, Geo, 4>), dim3((unsigned)n), dim3(256), 0, st, G, ang, cosv, sinv, sino,
                           img, acc, nty, nt, E);
    else
        hipLaunchKernelGGL((k_bp2d_tile<M, Geo, 16>), dim3((unsigned)n), dim3(1024), 0, st, G, ang, cosv, sinv, sino,
                           img, acc, nty, nt, E);
    return check_hip(hipGetLastError(), what);
}

}  // namespace vir
