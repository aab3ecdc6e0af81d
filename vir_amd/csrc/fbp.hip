// Filtered backprojection for gfx950: projection filtering as a direct
// convolution with the taps of a windowed ramp filter, and a pixel-driven
// weighted backprojection with linear interpolation (parallel beam, fan beam
// with a flat or an equiangular detector).
//
// Filtering.  filtration.filter_sino (filtration.py:267-329) zero-pads each
// row to z >= 2 nu, multiplies its rFFT by 2 H(f) (H the windowed ramp of
// ramp_filter / window_filter, filtration.py:4-264) and crops the inverse to
// nu samples.  H is real and even, so that is the linear convolution of the
// row with the symmetric kernel g = irfft(2 H) -- no wrap-around reaches the
// first nu outputs -- evaluated here as out[i] = sum_j w[j] row[j] g[|i - j|]
// from LDS copies of the row and the taps, in double.  The host designs g
// (and applies the equiangular (g/sin g)^2 correction to it).
//
// Backprojection.  Kak & Slaney's fan-beam formulas in the projector
// conventions of sys_mat/dd.py (view angle a, c = cos a, s = sin a; pixel
// centre (x, y); p = -s x + c y across the ray, o = c x + s y toward the
// source at DSO):
//   parallel : coordinate p,                                 weight 1
//   flat fan : virtual-detector coordinate DSO p / (DSO - o), weight (DSO / (DSO - o))^2
//   arc fan  : fan angle atan2(p, DSO - o),                  weight 1 / ((DSO - o)^2 + p^2)
// sampled by linear interpolation between bin centres (zero outside the
// detector; positions, weights and sums in double), times the caller's scale.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "vir_common.h"

namespace vir {

constexpr int kFbpMaxBins = 4096;

// Filtering: a Toeplitz product in float64.  A block computes OUT outputs of
// 512 / OUT rows: four consecutive ones of two rows a lane, OUT / 4 lanes a row.
// Its four waves take a quarter of every chunk of the sum and add their parts in
// wave order.  The taps g[|i - j|] of the tile lie in LDS as one float64 sequence,
// so moving to the next j shifts a lane's four taps by one: per j a tap and two
// row values are read for eight multiply-adds.  (One output a thread, converting
// a row value and a tap for every multiply-add: 169 us for 720 rows of 888; 41 us.)
// Rows of up to 128 values take the smallest OUT that holds them: 100000 rows of
// 16, 64, 128 values 27, 48, 98 us, as two rows of 256 outputs 129, 223, 333.
constexpr int kFfWaves = 4;

// place of tap w in LDS: every four taps are followed by an empty one, which
// puts the lanes' reads (four taps apart) on different banks
__device__ __forceinline__ int ff_at(int w) { return w + (w >> 2); }

template <int OUT>
__global__ __launch_bounds__(64 * kFfWaves) void k_fbp_filter(const float* __restrict__ sino, int64_t nrows, int nu,
                                                             const float* __restrict__ weight,
                                                             const float* __restrict__ taps, float* __restrict__ out,
                                                             int ntile) {
    constexpr int ROWS = 512 / OUT, CHUNK = OUT < 256 ? OUT : 512, TAPS = OUT + CHUNK, LPR = OUT / 4;
    constexpr int PITCH = CHUNK + (OUT < 256 ? 4 : 0);  // (rows that a wave reads together: different banks)
    __shared__ double h[TAPS + TAPS / 4 + 1];
    __shared__ double row[ROWS][PITCH];
    __shared__ double red[kFfWaves][ROWS * OUT];
    const int tid = threadIdx.x, sub = (tid & 63) % LPR, ra = 2 * ((tid & 63) / LPR);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i0 = (int)(blockIdx.x % ntile) * OUT;
    const int64_t r0 = (int64_t)(blockIdx.x / ntile) * ROWS;
    double acc[2][4] = {};
    for (int jc = 0; jc < nu; jc += CHUNK) {
        __syncthreads();
        // h[w] = g[|i0 + w - (jc + CHUNK)|], w = 0 .. TAPS - 1: the tap of output
        // i0 + i and input jc + j lies at w = CHUNK + i - j
        for (int w = tid; w < TAPS; w += 64 * kFfWaves) {
            const int k = abs(i0 + w - (jc + CHUNK));
            h[ff_at(w)] = k < nu ? (double)taps[k] : 0.0;
        }
        for (int e = tid; e < ROWS * CHUNK; e += 64 * kFfWaves) {
            const int r = e / CHUNK, j = jc + e % CHUNK;
            float x = 0.0f;
            if (r0 + r < nrows && j < nu) {
                x = sino[(r0 + r) * nu + j];
                if (weight) x = x * weight[j];
            }
            row[r][e % CHUNK] = (double)x;
        }
        __syncthreads();
        // this wave's quarter, four inputs at a time: taps w - 3 .. w + 3 of
        // w = CHUNK + 4 sub - j, of which the upper three stay from before
        const int ja = wave * (CHUNK / kFfWaves), jb = min(ja + CHUNK / kFfWaves, nu - jc);
        if (ja >= jb) continue;
        const double* hl = h + ff_at(CHUNK + 4 * sub - ja);
        double t0 = hl[0], t1 = hl[1], t2 = hl[2], t3 = hl[3];
        for (int j = ja; j < jb; j += 4, hl -= 5) {
            const double s0 = hl[-5], s1 = hl[-4], s2 = hl[-3], s3 = hl[-2];  // w - 4 .. w - 1
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const double* x = row[ra + r] + j;
                const double x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
                const auto f = [](double x, double y, double z) { return __builtin_fma(x, y, z); };
                acc[r][0] = f(x3, s1, f(x2, s2, f(x1, s3, f(x0, t0, acc[r][0]))));
                acc[r][1] = f(x3, s2, f(x2, s3, f(x1, t0, f(x0, t1, acc[r][1]))));
                acc[r][2] = f(x3, s3, f(x2, t0, f(x1, t1, f(x0, t2, acc[r][2]))));
                acc[r][3] = f(x3, t0, f(x2, t1, f(x1, t2, f(x0, t3, acc[r][3]))));
            }
            t0 = s0; t1 = s1; t2 = s2; t3 = s3;
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][(ra + r) * OUT + 4 * sub + q] = acc[r][q];
    __syncthreads();
    for (int e = tid; e < ROWS * OUT; e += 64 * kFfWaves) {
        const int64_t r = r0 + e / OUT;
        const int i = i0 + e % OUT;
        if (r >= nrows || i >= nu) continue;
        double s = red[0][e];
#pragma unroll
        for (int w = 1; w < kFfWaves; ++w) s += red[w][e];
        out[r * nu + i] = (float)s;
    }
}

struct FbpGeo {
    int nx, ny, nu, na, mode;
    float d, DSO;
    double c0, inv_du;  // filter-domain coordinate of bin 0's centre, 1 / bin spacing
    float scale;
};

// 1/x to float64 rounding: the hardware's reciprocal (relative error e = 2^-24)
// times 1 + e + e^2
__device__ __forceinline__ double fbp_rcp(double x) {
    const double r = __builtin_amdgcn_rcp(x), e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// Backprojection: geometry and interpolation in double (the filtered
// projections are rough -- ramp-filtered noise -- so the sampling position must
// not round).  A block takes 16 x 16 pixels, a 2 x 2 block a lane; wave w of its
// NW takes views w, w + NW, ... and the waves' sums are added in wave order.
// Per view the constants that the tile shares are formed by one lane.
//
// Equiangular detector: with (a, b) a pixel's coordinates along and across the
// ray through the tile's centre, its fan angle is the centre's plus atan(t), t =
// b / a, and its weight 1/L^2 = 1 / (a^2 (1 + t^2)).  A tile is small against
// its distance, so short series do: for |t| <= 0.06 (FAR = 1) to t^11 and t^12,
// for |t| <= 0.02 (FAR = 2) to t^7 and t^8.  The angle's next terms, t^13/13 and
// t^9/9, are below 1.1e-17 and 5.7e-17 rad, the weight's, t^14 and t^10, below 8e-18
// and 1.1e-17 of it: with 10^4 bins a radian 6e-13 bin, where a float64 position of
// 1000 bins rounds by 1e-13.  Nearer sources (FAR = 0) take atan2.
// Bound by float64 VALU work.  An atan2 and a division in double for every
// pixel and view took 820 us at 512^2, 720 views of 888; FAR = 1 300 us, FAR = 2
// 280 us.
constexpr double kFbpFar1 = 0.06, kFbpFar2 = 0.02;

template <int MODE, int FAR, int NW>
__global__ __launch_bounds__(64 * NW) void k_fbp_bp(FbpGeo G, const float* __restrict__ cs,
                                                    const float* __restrict__ sn, const float* __restrict__ q,
                                                    float* __restrict__ img, int accumulate, int nty) {
    constexpr bool ARC = MODE == 2 && FAR > 0;
    __shared__ double cv[NW][64][4];
    __shared__ double red[NW][256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int bx = (int)(blockIdx.x / nty) * 16, by = (int)(blockIdx.x % nty) * 16;
    const double d = G.d, DSO = G.DSO;
    // tile centre, and this lane's pixels from it
    const double xc = d * ((double)(bx + 8) - 0.5 * (double)G.nx), yc = d * ((double)(by + 8) - 0.5 * (double)G.ny);
    const double dx = d * ((double)(2 * (lane >> 3)) - 7.5), dy = d * ((double)(2 * (lane & 7)) - 7.5);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int g = 0; g < G.na; g += 64 * NW) {
        {
            const int ia = min(g + NW * lane + wave, G.na - 1);
            const double c = cs[ia], s = sn[ia];
            const double p = -s * xc + c * yc, o = DSO - (c * xc + s * yc);
            double* v = cv[wave][lane];
            if (ARC) {
                const double L = sqrt(p * p + o * o), ce = o / L, se = p / L;
                v[0] = c * ce + s * se;   // a = L - v0 x + v1 y, b = v1 x + v0 y
                v[1] = c * se - s * ce;
                v[2] = L;
                v[3] = (atan2(p, o) - G.c0) * G.inv_du;
            } else {
                v[0] = c;
                v[1] = s;
                v[2] = p;
                v[3] = o;
            }
            // a view without a finite angle: four bins off the detector's start,
            // where it adds nothing (flat fan and atan2: tested per pixel)
            if ((MODE == 0 || ARC) && !(fabs(p) + fabs(o) < (double)VIR_INF)) {
                v[0] = v[1] = 0.0;
                v[2] = ARC ? 1.0 : G.c0 - 4.0 / G.inv_du;
                v[3] = ARC ? -4.0 : 0.0;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a wave's LDS accesses are in order
        const int nl = min(64, (G.na - g - wave + NW - 1) / NW);
        for (int l = 0; l < nl; ++l) {
            const double v0 = cv[wave][l][0], v1 = cv[wave][l][1], v2 = cv[wave][l][2], v3 = cv[wave][l][3];
            const float* __restrict__ row = q + (int64_t)(g + NW * l + wave) * G.nu;
            double w[4], fr[4];
            float ya[4], yb[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double x = k & 2 ? dx + d : dx, y = k & 1 ? dy + d : dy;
                double tf;
                if (ARC) {
                    const double a = __builtin_fma(v1, y, __builtin_fma(-v0, x, v2)), b = __builtin_fma(v0, y, v1 * x);
                    const double r = fbp_rcp(a), t = b * r, u = t * t;
                    const auto f = [&](double z, double cst) { return __builtin_fma(z, u, cst); };
                    const double a7 = FAR == 2 ? -1.0 / 7.0 : f(f(-1.0 / 11.0, 1.0 / 9.0), -1.0 / 7.0);
                    const double at = t * f(f(f(a7, 1.0 / 5.0), -1.0 / 3.0), 1.0);
                    const double w4 = FAR == 2 ? 1.0 : f(f(1.0, -1.0), 1.0);
                    w[k] = (r * r) * f(f(f(f(w4, -1.0), 1.0), -1.0), 1.0);
                    tf = __builtin_fma(at, G.inv_du, v3);
                } else {
                    const double p = __builtin_fma(v0, y, __builtin_fma(-v1, x, v2));
                    const double o = __builtin_fma(-v1, y, __builtin_fma(-v0, x, v3));
                    double coord = p;
                    w[k] = 1.0;
                    if (MODE == 1) {
                        const double m = DSO * fbp_rcp(o);
                        coord = m * p;
                        w[k] = m * m;
                    } else if (MODE == 2) {
                        coord = atan2(p, o);
                        w[k] = 1.0 / (o * o + p * p);
                    }
                    tf = (coord - G.c0) * G.inv_du;
                }
                const double fl = floor(tf);
                fr[k] = tf - fl;
                int j = (int)fl;  // saturates; outside the detector both ends read as zero
                if (MODE > 0 && !ARC) {  // a pixel on the source's plane has no position
                    const bool ok = fl >= -1.0 && fl <= (double)G.nu - 1.0;
                    fr[k] = ok ? fr[k] : 0.0;
                    w[k] = ok ? w[k] : 0.0;
                    j = ok ? j : -2;
                }
                j = min(max(j, -2), G.nu);
                ya[k] = row[min(max(j, 0), G.nu - 1)];
                yb[k] = row[min(max(j, -1) + 1, G.nu - 1)];
                ya[k] = (unsigned)j < (unsigned)G.nu ? ya[k] : 0.0f;
                yb[k] = (unsigned)(j + 1) < (unsigned)G.nu ? yb[k] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                acc[k] = __builtin_fma(w[k], __builtin_fma(fr[k], (double)yb[k], (1.0 - fr[k]) * (double)ya[k]), acc[k]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) red[wave][64 * k + lane] = acc[k];
    __syncthreads();
    for (int i = threadIdx.x; i < 256; i += 64 * NW) {
        const int x = i >> 4, y = i & 15;  // consecutive threads, consecutive pixels
        const int slot = 64 * (2 * (x & 1) + (y & 1)) + 8 * (x >> 1) + (y >> 1);
        if (bx + x >= G.nx || by + y >= G.ny) continue;
        double s = red[0][slot];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += red[w][slot];
        const int64_t o = (int64_t)(bx + x) * G.ny + by + y;
        float r = (float)s * G.scale;
        if (accumulate) r += img[o];
        img[o] = r;
    }
}

template <int MODE, int FAR>
static void fbp_bp(const FbpGeo& G, const float* cosv, const float* sinv, const float* q, float* img, int acc,
                   hipStream_t st) {
    const int nty = (G.ny + 15) / 16;
    const int64_t n = (int64_t)((G.nx + 15) / 16) * nty;
    // sixteen waves share a tile's views where the tiles alone leave CUs idle
    if (n >= 1024)
        hipLaunchKernelGGL((k_fbp_bp<MODE, FAR, 4>), dim3((unsigned)n), dim3(256), 0, st, G, cosv, sinv, q, img, acc, nty);
    else
        hipLaunchKernelGGL((k_fbp_bp<MODE, FAR, 16>), dim3((unsigned)n), dim3(1024), 0, st, G, cosv, sinv, q, img, acc, nty);
}

}  // namespace vir

using namespace vir;

extern "C" {

int vir_fbp_filter(const float* sino, int64_t nrows, int32_t nu, const float* weight, const float* taps, float* out,
                   void* stream) {
    if (nrows < 0 || nu < 1) return fail_arg("nrows must be >= 0 and nu >= 1");
    if (nu > kFbpMaxBins) return fail_arg("nu exceeds 4096 detector bins");
    if (nrows == 0) return VIR_OK;
    if (!sino || !taps || !out) return fail_arg("NULL pointer argument");
    if (sino == out) return fail_arg("in-place filtering is not supported");
    hipStream_t st = as_stream(stream);
    const auto run = [&](auto width) {
        constexpr int OUT = decltype(width)::value, ROWS = 512 / OUT;
        const int ntile = (nu + OUT - 1) / OUT;
        const int64_t most = kLaunchThreads / (64 * kFfWaves) / ntile * ROWS;  // rows a launch takes
        for (int64_t r = 0; r < nrows; r += most) {
            const int64_t n = std::min(most, nrows - r);
            hipLaunchKernelGGL(k_fbp_filter<OUT>, dim3((unsigned)((n + ROWS - 1) / ROWS * ntile)), dim3(64 * kFfWaves), 0,
                               st, sino + r * nu, n, nu, weight, taps, out + r * nu, ntile);
        }
    };
    if (nu <= 32) run(std::integral_constant<int, 32>{});
    else if (nu <= 64) run(std::integral_constant<int, 64>{});
    else if (nu <= 128) run(std::integral_constant<int, 128>{});
    else run(std::integral_constant<int, 256>{});
    return check_hip(hipGetLastError(), "vir_fbp_filter launch");
}

int vir_fbp_bp(const vir_dd_geom* geom, const float* cosv, const float* sinv, const float* q, float* img,
               float scale, uint32_t flags, void* stream) {
    if (!geom) return fail_arg("geometry is NULL");
    if (geom->mode < 0 || geom->mode > 2) return fail_arg("mode must be 0 (par), 1 (fan flat) or 2 (fan arc)");
    if (geom->nx < 1 || geom->ny < 1 || geom->nu < 1 || geom->na < 0) return fail_arg("bad sizes");
    if (!(geom->d_pix > 0.0f) || !(geom->du > 0.0f)) return fail_arg("spacings must be > 0");
    if (geom->mode > 0 && !(geom->DSO > 0.0f && geom->DSD > 0.0f)) return fail_arg("DSO and DSD must be > 0");
    if (!img || (geom->na > 0 && (!cosv || !sinv || !q))) return fail_arg("NULL pointer argument");
    FbpGeo G;
    G.nx = geom->nx; G.ny = geom->ny; G.nu = geom->nu; G.na = geom->na; G.mode = geom->mode;
    G.d = geom->d_pix; G.DSO = geom->DSO; G.scale = scale;
    // bin-0 centre and spacing in the filter domain (detector, virtual
    // detector through the isocentre, or fan angle)
    const double u0 = (double)geom->du * (0.5 - 0.5 * geom->nu + (double)geom->su);
    double f = 1.0;
    if (geom->mode == 1) f = (double)geom->DSO / geom->DSD;
    if (geom->mode == 2) f = 1.0 / geom->DSD;
    G.c0 = u0 * f;
    G.inv_du = 1.0 / ((double)geom->du * f);
    hipStream_t st = as_stream(stream);
    const int acc = (flags & VIR_ACCUMULATE) ? 1 : 0;
    // |t| of a tile: its half-diagonal over its least distance to the source
    const double half = 0.70711 * 15.0 * (double)G.d;  // (the source ahead of every tile, padding included)
    const double dist = (double)G.DSO - 0.5 * std::sqrt((double)(G.nx + 32) * (G.nx + 32) + (double)(G.ny + 32) * (G.ny + 32)) * G.d;
    const double t = dist > 0.0 ? half / dist : 1.0;
    if (G.mode == 0) fbp_bp<0, 0>(G, cosv, sinv, q, img, acc, st);
    else if (G.mode == 1) fbp_bp<1, 0>(G, cosv, sinv, q, img, acc, st);
    else if (t <= kFbpFar2) fbp_bp<2, 2>(G, cosv, sinv, q, img, acc, st);
    else if (t <= kFbpFar1) fbp_bp<2, 1>(G, cosv, sinv, q, img, acc, st);
    else fbp_bp<2, 0>(G, cosv, sinv, q, img, acc, st);
    return check_hip(hipGetLastError(), "vir_fbp_bp launch");
}

}  // extern "C"
