// Total-variation denoising by Chambolle's projection algorithm
// (A. Chambolle, "An algorithm for total variation minimization and
// applications", J. Math. Imaging Vis. 20 (2004) 89-97, eq. (9)):
//
//   u = argmin_u ||u - g||^2 / 2 + w TV(u),  TV(u) = sum_i |(grad u)_i|,
//
// grad = forward differences along each axis (zero at the last index),
// div = -grad^T.  In the dual variable q = w p:
//
//   v = div q - g
//   q <- (q + tau grad v) / (1 + (tau / w) |grad v|)
//   u  = g - div q
//
// One iteration is two launches over the voxels (grid-stride, 256 threads):
// the residual v into a scratch image, then the dual step, in place on q
// (each q element is read and written by its own thread; v is not written).
// q holds one plane per axis, plane a at offset a * n; its values at an
// axis' last index are taken as zero.  The step also keeps the largest
// |q_new - q_old| per block for the host's stopping rule.
#include <algorithm>
#include <cmath>

#include "vir_common.h"

namespace vir {

constexpr int kTvdBlocks = 2048;  // VIR_TV_WORK

struct TvdShape {
    int64_t n;           // voxels
    int n0, n1, n2;      // sizes along axes 0, 1, 2 (1 for missing axes)
    int64_t s0, s1;      // strides of axes 0 and 1 (axis 2: 1)
};

template <int ND>
__device__ __forceinline__ void tvd_coords(const TvdShape& S, int64_t j, int (&i)[3]) {
    i[2] = (int)(j % S.n2);
    const int64_t r = j / S.n2;
    i[1] = (int)(r % S.n1);
    i[0] = (int)(r / S.n1);
}

// v = sign (div q - g)
template <int ND>
__global__ __launch_bounds__(256) void k_tvd_residual(TvdShape S, const float* __restrict__ q,
                                                     const float* __restrict__ g, float sign,
                                                     float* __restrict__ v) {
    const int nn[3] = {S.n0, S.n1, S.n2};
    const int64_t st[3] = {S.s0, S.s1, 1};
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < S.n;
         j += (int64_t)gridDim.x * blockDim.x) {
        int i[3];
        tvd_coords<ND>(S, j, i);
        float d = 0.0f;
#pragma unroll
        for (int a = 0; a < ND; ++a) {
            const float* __restrict__ qa = q + a * S.n;
            if (i[a] < nn[a] - 1) d += qa[j];
            if (i[a] > 0) d -= qa[j - st[a]];
        }
        v[j] = sign * (d - g[j]);
    }
}

template <int ND>
__global__ __launch_bounds__(256) void k_tvd_step(TvdShape S, const float* __restrict__ v, float* __restrict__ q,
                                                 float tau, float tau_w, float* __restrict__ dmax) {
    const int nn[3] = {S.n0, S.n1, S.n2};
    const int64_t st[3] = {S.s0, S.s1, 1};
    float m = 0.0f;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < S.n;
         j += (int64_t)gridDim.x * blockDim.x) {
        int i[3];
        tvd_coords<ND>(S, j, i);
        const float vj = v[j];
        float gr[ND];
        float n2 = 0.0f;
#pragma unroll
        for (int a = 0; a < ND; ++a) {
            gr[a] = i[a] < nn[a] - 1 ? v[j + st[a]] - vj : 0.0f;
            n2 += gr[a] * gr[a];
        }
        const float den = 1.0f + tau_w * sqrtf(n2);
#pragma unroll
        for (int a = 0; a < ND; ++a) {
            float* __restrict__ qa = q + a * S.n;
            const float old = qa[j];
            const float nw = (old + tau * gr[a]) / den;
            qa[j] = nw;
            m = fmaxf(m, fabsf(nw - old));
        }
    }
    if (!dmax) return;
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_down(m, off, 64));
    __shared__ float red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) dmax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(256) void k_tvd_max(float* __restrict__ dmax, int nblk) {
    __shared__ float red[256];
    float m = 0.0f;
    for (int k = threadIdx.x; k < nblk; k += 256) m = fmaxf(m, dmax[k]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) dmax[0] = red[0];
}

// ----------------------------------------------- several iterations a pass
//
// The two launches above read and write 12 values a voxel and iteration (3-D)
// and are bound by HBM: 247 us an iteration at 256^3.  k_tvd_march reads q and
// g once, runs K iterations and writes q once, into a second array.
//
// At 256^3 two iterations take 150 us, 600 MB of HBM traffic (380 read with
// the tiles' margins; 36 B a voxel, where q and g read and q written once are 28):
// 4.0 of the 5.2 TB/s of a copy.  With one iteration a pass a launch takes longer
// still (170 us), with two or four rows a lane instead of three 50 iterations take
// 4.5 or 9.6 ms (spills) against 3.99, and without the XCD placement 4.3.
//
// A wave covers 64 voxels along the last axis (lane = voxel) and marches along
// axis 0; in 3-D each lane holds R rows along axis 1 and the G waves of a
// block lie one after another along it.  Iteration stages are pipelined: at
// step s stage k takes plane x_k = xs + s - 2k of q^k, forms v there and, with
// v of plane x_k - 1 from the step before, q^(k+1) of plane x_k - 1, which stage
// k + 1 takes at the next step.  So the stages of a step are independent, and
// a step has one barrier (the rows at the waves' ends pass through LDS).  A
// tile's outer K voxels and rows are recomputed by its neighbours; a block
// marches over a chunk of planes with 2K - 1 planes of lead.
//
// The arithmetic of a voxel is that of the two-launch kernels, operation by
// operation; the square root and the quotients (old + tau grad) / den are
// correctly rounded by residuals (Markstein) instead of the general sequences,
// 40 % fewer VALU instructions.
//
// Voxels outside the image hold q = 0, as does q at an axis' last index (the
// start value zero stays zero there), which stands for the two-launch kernels'
// tests of the index.
__device__ __forceinline__ float tvd_below(float x) {  // of the lane below (0 into lane 0)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float tvd_above(float x) {  // of the lane above (0 into lane 63)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}

// Correctly rounded square root: the hardware's (1 ulp), then whichever
// neighbour the residuals pick.  (Arguments below 2^-96, where residuals
// underflow, add nothing to 1 + tau_w sqrt.)
__device__ __forceinline__ float tvd_sqrt(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __int_as_float(__float_as_int(s) - 1), hi = __int_as_float(__float_as_int(s) + 1);
    float r = __builtin_fmaf(-lo, s, x) <= 0.0f ? lo : s;
    return __builtin_fmaf(-hi, s, x) > 0.0f ? hi : r;
}

template <int ND, int K, int R, int G>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(4))) void k_tvd_march(TvdShape S, const float* __restrict__ qi,
                                                     float* __restrict__ qo, const float* __restrict__ g, float tau,
                                                     float tau_w, float* __restrict__ dmax, int chunk, int nty,
                                                     int ntz) {
    static_assert(ND == 3 || R == 1, "rows are axis 1 of a volume");
    constexpr int NC = ND;
    // rows at the ends of each wave's block: q's axis-1 component of the last
    // row (for the wave after), v of the first row (for the wave before)
    __shared__ float eq[ND == 3 ? 2 : 1][K][G][64], ev[ND == 3 ? 2 : 1][K][G][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nz = ND == 3 ? S.n2 : S.n1, ny = ND == 3 ? S.n1 : 1;
    // 3-D: the block's tile; 2-D: each wave's own strip and chunk
    int t = (int)xcd_remap(blockIdx.x, gridDim.x);
    if (ND == 2) t = t * G + wave;
    const int z = (t % ntz) * (64 - 2 * K) - K + lane;
    t /= ntz;
    const int y0 = ND == 3 ? (t % nty) * (G * R - 2 * K) - K + wave * R : 0;
    if (ND == 3) t /= nty;
    const int xa = t * chunk, xb = min(xa + chunk, S.n0);  // planes written
    const bool zin = z >= 0 && z < nz, zout = zin && lane >= K && lane < 64 - K;
    int64_t off[R];
    bool in[R], out[R], my[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = y0 + r;
        in[r] = zin && y >= 0 && y < ny;
        out[r] = zout && in[r] && (ND == 2 || (wave * R + r >= K && wave * R + r < G * R - K));
        my[r] = in[r] && y < ny - 1;
        off[r] = (ND == 3 ? (int64_t)y * S.s1 : 0) + z;
    }
    const bool mz = z < nz - 1;

    // q^k at stage k's plane and the one before, in turn (qs[s & 1] holds step
    // s's planes); v of the plane before; g of the planes x, x - 2, .. of one
    // parity; the next plane, loaded a step ahead
    float qs[2][K][NC][R], vp[K][R], gs[2][K][R], nq[NC][R], ng[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < K; ++k) {
            vp[k][r] = gs[0][k][r] = gs[1][k][r] = 0.0f;
#pragma unroll
            for (int a = 0; a < NC; ++a) qs[0][k][a][r] = qs[1][k][a][r] = 0.0f;
        }
    const auto load = [&](int x) {
        const bool px = x >= 0 && x < S.n0;
        const int64_t base = (int64_t)x * S.s0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int a = 0; a < NC; ++a) nq[a][r] = px && in[r] ? qi[a * S.n + base + off[r]] : 0.0f;
            ng[r] = px && in[r] ? g[base + off[r]] : 0.0f;
        }
    };
    // stage 0 starts K planes before the first one written: v of that plane
    // and every later stage's first plane are garbage that no output uses
    const int xs = xa - K, steps = xb - xs + 2 * K - 1;
    float m = 0.0f;
    const auto step = [&](int s, float (&qc)[K][NC][R], float (&qp)[K][NC][R], float (&gf)[K][R], int p) {
        const int x = xs + s;
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int a = 0; a < NC; ++a) qc[0][a][r] = nq[a][r];
#pragma unroll
            for (int i = K - 1; i > 0; --i) gf[i][r] = gf[i - 1][r];
            gf[0][r] = ng[r];
        }
        if (s + 1 < steps) load(x + 1);
        if (ND == 3) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                eq[p][k][wave][lane] = qc[k][1][R - 1];
                ev[p][k][wave][lane] = vp[k][0];
            }
            __syncthreads();
        }
        // the last stage first: stage k leaves its result where stage k + 1 had
        // its plane before, for the next step
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const int xk = x - 2 * k;
            const bool mx = xk >= 1 && xk < S.n0;  // plane x_k - 1 has a next one
            const bool written = k == K - 1 && xk - 1 >= xa && xk - 1 < xb;
            float yq = 0.0f, yv = 0.0f;
            if (ND == 3) {
                if (wave > 0) yq = eq[p][k][wave - 1][lane];
                if (wave < G - 1) yv = ev[p][k][wave + 1][lane];
            }
            float nx[NC][R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float d = qc[k][0][r] - qp[k][0][r];
                if (ND == 3) {
                    d += qc[k][1][r];
                    d -= r > 0 ? qc[k][1][r > 0 ? r - 1 : 0] : yq;
                }
                d += qc[k][NC - 1][r];
                d -= tvd_below(qc[k][NC - 1][r]);
                const float v = d - gf[k][r], v0 = vp[k][r];
                const float vz = tvd_above(v0);  // every lane takes part
                float gr[NC], n2;
                gr[0] = mx && in[r] ? v - v0 : 0.0f;
                n2 = gr[0] * gr[0];
                if (ND == 3) {
                    gr[1] = my[r] ? (r < R - 1 ? vp[k][r < R - 1 ? r + 1 : r] : yv) - v0 : 0.0f;
                    n2 += gr[1] * gr[1];
                }
                gr[NC - 1] = mz && in[r] ? vz - v0 : 0.0f;
                n2 += gr[NC - 1] * gr[NC - 1];
                float den = 1.0f + tau_w * tvd_sqrt(n2);
                den = den == VIR_INF ? 3.4028235e38f : den;  // quotients by infinity: zero
                float rd = __builtin_amdgcn_rcpf(den);
                rd = __builtin_fmaf(__builtin_fmaf(-den, rd, 1.0f), rd, rd);
#pragma unroll
                for (int a = 0; a < NC; ++a) {
                    const float num = qp[k][a][r] + tau * gr[a], q0 = num * rd;
                    nx[a][r] = __builtin_fmaf(__builtin_fmaf(-q0, den, num), rd, q0);
                }
                vp[k][r] = v;  // rows in order: the row before has used v0
            }
            if (written) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int a = 0; a < NC; ++a)
                        if (out[r]) {
                            qo[a * S.n + (int64_t)(xk - 1) * S.s0 + off[r]] = nx[a][r];
                            if (dmax) m = fmaxf(m, fabsf(nx[a][r] - qp[k][a][r]));
                        }
            }
            if (k + 1 < K) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int a = 0; a < NC; ++a) qp[k + 1 < K ? k + 1 : k][a][r] = nx[a][r];
            }
        }
    };
    load(xs);
    for (int s = 0; s < steps; s += 2) {
        step(s, qs[0], qs[1], gs[0], 0);
        if (s + 1 < steps) step(s + 1, qs[1], qs[0], gs[1], 1);
    }
    if (!dmax) return;
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_down(m, o, 64));
    // non-negative floats compare as their bits do
    if (lane == 0) atomicMax((int*)dmax + (blockIdx.x * G + wave) % kTvdBlocks, __float_as_int(m));
}

__global__ __launch_bounds__(256) void k_tvd_zero(float* __restrict__ dmax) {
    for (int i = threadIdx.x; i < kTvdBlocks; i += 256) dmax[i] = 0.0f;
}

// Tiles, planes a chunk and chunks of a pass of K iterations.  A volume's blocks
// (eight waves of three rows) run two to a CU; its chunks of planes are as long
// as 512 blocks allow, since every chunk adds 3K - 1 planes of lead (400 blocks:
// 4.27 ms for 50 iterations at 256^3, against 3.99).  An image's waves work
// alone: 2048 of them.
struct TvdPlan {
    int ntz, nty, chunk;
    int64_t n;  // blocks (3-D) or waves (2-D)
};

template <int ND, int K>
static TvdPlan tvd_plan(const TvdShape& S) {
    constexpr int R = ND == 3 ? 3 : 1, G = ND == 3 ? 8 : 4;
    const int nz = ND == 3 ? S.n2 : S.n1, ny = ND == 3 ? S.n1 : 1;
    TvdPlan P;
    P.ntz = (nz + 63 - 2 * K) / (64 - 2 * K);
    P.nty = ND == 3 ? (ny + G * R - 2 * K - 1) / (G * R - 2 * K) : 1;
    const int64_t tiles = (int64_t)P.ntz * P.nty, want = std::max<int64_t>(1, (ND == 3 ? 512 : 2048) / tiles);
    P.chunk = (int)std::max<int64_t>(ND == 3 ? 8 : 16, (S.n0 + want - 1) / want);
    P.n = tiles * ((S.n0 + P.chunk - 1) / P.chunk);
    return P;
}

// Iterations on two copies of q in turn; *cur: the copy that holds q.
template <int ND, int K>
static void tvd_march(const TvdShape& S, const float* g, float* const* q, int32_t* cur, float weight, float tau,
                      float* dmax, hipStream_t st) {
    constexpr int R = ND == 3 ? 3 : 1, G = ND == 3 ? 8 : 4;
    const TvdPlan P = tvd_plan<ND, K>(S);
    if (dmax) hipLaunchKernelGGL(k_tvd_zero, dim3(1), dim3(256), 0, st, dmax);
    hipLaunchKernelGGL((k_tvd_march<ND, K, R, G>), dim3((unsigned)(ND == 3 ? P.n : (P.n + G - 1) / G)), dim3(64 * G), 0,
                       st, S, q[*cur], q[1 - *cur], g, tau, tau / weight, dmax, P.chunk, P.nty, P.ntz);
    if (dmax) hipLaunchKernelGGL(k_tvd_max, dim3(1), dim3(256), 0, st, dmax, kTvdBlocks);
    *cur = 1 - *cur;
}

// Whether a pass of K iterations is faster than K times two launches.  It marches
// plane by plane, in serial, and its lanes lie along the last axis, so small
// and thin images are better off with the launches: those take about 3 us and
// 11.5 (images 8) a million voxels an iteration, at least 8 (7.2); a pass 1.65
// us a plane up to 256 blocks, 2.35 beyond (images 0.95), and at least 9 us a
// million voxels.  Launches | passes for ten iterations in us: 64^3 87 | 109, 512
// x 512 x 1 83 | 362, x 4 148 | 368, x 16 478 | 367, 256^3 2499 | 759, 200000 x 4 111 | 189,
// 2048^2 370 | 96.  Of 644 sizes measured three take up to 1.2 times the other
// way's time.
template <int ND, int K>
static bool tvd_pays(const TvdShape& S) {
    const TvdPlan P = tvd_plan<ND, K>(S);
    if (P.n * 512 > kLaunchThreads) return false;
    const double m = 1e-6 * (double)S.n, planes = std::min(P.chunk, S.n0) + 3 * K - 1;
    if (ND == 2) return planes * 0.95 <= K * std::max(7.2, 3.0 + 8.0 * m);
    return std::max(planes * (P.n <= 256 ? 1.65 : 2.35), 9.0 * m) <= K * std::max(8.0, 3.0 + 11.5 * m);
}

template <int ND, int K>
static int tvd_pair(const TvdShape& S, const float* g, float* const* q, int32_t* cur, float weight, float tau,
                    int iters, float* dmax, hipStream_t st) {
    for (; iters >= K; iters -= K) tvd_march<ND, K>(S, g, q, cur, weight, tau, iters == K ? dmax : nullptr, st);
    for (; iters > 0; --iters) tvd_march<ND, 1>(S, g, q, cur, weight, tau, iters == 1 ? dmax : nullptr, st);
    return check_hip(hipGetLastError(), "vir_tv_chambolle_pair launch");
}

template <int ND>
static int tvd_run(const TvdShape& S, const float* g, float* q, float* v, float* u, float weight, float tau,
                   int iters, float* dmax, hipStream_t st) {
    const int64_t want = (S.n + 255) / 256;
    const int nblk = (int)(want < kTvdBlocks ? want : kTvdBlocks);
    for (int it = 0; it < iters; ++it) {
        hipLaunchKernelGGL(k_tvd_residual<ND>, dim3(nblk), dim3(256), 0, st, S, q, g, 1.0f, v);
        float* dm = (dmax && it == iters - 1) ? dmax : nullptr;
        hipLaunchKernelGGL(k_tvd_step<ND>, dim3(nblk), dim3(256), 0, st, S, v, q, tau, tau / weight, dm);
    }
    if (dmax && iters > 0) hipLaunchKernelGGL(k_tvd_max, dim3(1), dim3(256), 0, st, dmax, nblk);
    if (u) hipLaunchKernelGGL(k_tvd_residual<ND>, dim3(nblk), dim3(256), 0, st, S, q, g, -1.0f, u);
    return check_hip(hipGetLastError(), "vir_tv_chambolle launch");
}

}  // namespace vir

using namespace vir;

static int tvd_args(int32_t ndim, int32_t nx, int32_t ny, int32_t nz, float weight, float tau, int32_t iters,
                    TvdShape& S) {
    if (ndim < 1 || ndim > 3) return fail_arg("ndim must be 1, 2 or 3");
    if (nx < 1 || ny < 1 || nz < 1) return fail_arg("sizes must be >= 1");
    if ((ndim < 2 && ny != 1) || (ndim < 3 && nz != 1)) return fail_arg("sizes of missing axes must be 1");
    if (!(weight > 0.0f) || !std::isfinite(weight)) return fail_arg("weight must be > 0");
    if (!(tau > 0.0f) || !std::isfinite(tau)) return fail_arg("tau must be > 0");
    if (iters < 0) return fail_arg("iters must be >= 0");
    S.n0 = nx; S.n1 = ny; S.n2 = nz;
    S.n = (int64_t)nx * ny * nz;
    S.s1 = nz;
    S.s0 = (int64_t)ny * nz;
    return VIR_OK;
}

extern "C" {

int vir_tv_chambolle(int32_t ndim, int32_t nx, int32_t ny, int32_t nz, const float* g, float* q, float* v,
                     float* u, float weight, float tau, int32_t iters, float* dmax, void* stream) {
    TvdShape S;
    if (const int rc = tvd_args(ndim, nx, ny, nz, weight, tau, iters, S)) return rc;
    if (!g || !q || (iters > 0 && !v)) return fail_arg("NULL pointer argument");
    hipStream_t st = as_stream(stream);
    if (ndim == 1) return tvd_run<1>(S, g, q, v, u, weight, tau, iters, dmax, st);
    if (ndim == 2) return tvd_run<2>(S, g, q, v, u, weight, tau, iters, dmax, st);
    return tvd_run<3>(S, g, q, v, u, weight, tau, iters, dmax, st);
}

int vir_tv_pair_pays(int32_t ndim, int32_t nx, int32_t ny, int32_t nz) {
    TvdShape S;
    if (ndim < 2 || tvd_args(ndim, nx, ny, nz, 1.0f, 1.0f, 1, S)) return 0;
    return ndim == 2 ? tvd_pays<2, 5>(S) : tvd_pays<3, 2>(S);
}

int vir_tv_chambolle_pair(int32_t ndim, int32_t nx, int32_t ny, int32_t nz, const float* g, float* q0, float* q1,
                          int32_t* cur, float weight, float tau, int32_t iters, float* dmax, void* stream) {
    TvdShape S;
    if (const int rc = tvd_args(ndim, nx, ny, nz, weight, tau, iters, S)) return rc;
    if (ndim < 2) return fail_arg("ndim must be 2 or 3");
    if (!g || !q0 || !q1 || !cur) return fail_arg("NULL pointer argument");
    if (*cur != 0 && *cur != 1) return fail_arg("*cur must be 0 or 1");
    float* q[2] = {q0, q1};
    hipStream_t st = as_stream(stream);
    if (ndim == 2) return tvd_pair<2, 5>(S, g, q, cur, weight, tau, iters, dmax, st);
    return tvd_pair<3, 2>(S, g, q, cur, weight, tau, iters, dmax, st);
}

}  // extern "C"
