// Sums over all nodes of an iterate: the theta step, the explicit objective with its KKT residual,
// and the reconstruction error.  A grid of at most READ_BLOCKS workgroups strides over the nodes,
// each thread keeping its sums in registers; one more workgroup adds the workgroups' partials
// and writes the few results to pinned host memory.  With one partial row per 256 nodes and the
// rest of the sum on the host, the theta step at T = 1e7, K = 3 moved 1.9 MB of partials and took
// 400 us, the objective 210 us; now 80 and 90 us, against 58 us for their bytes at the copy rate.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "util_kernels.h"

namespace pasc {

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(PASC_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));     \
    } while (0)

constexpr int RNTH = 256;
constexpr int FINISH_WAVES = 8;

// The workgroup's sums of v to part[v * gridDim.x + block]; a value of index `mx` is a maximum.
template <int NV>
__device__ __forceinline__ void put_partials(double (&v)[NV], int mx, double *lds, double *part) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const double s = i == mx ? wave_max(v[i]) : wave_sum(v[i]);
        if (lane == 0) lds[i * (RNTH / WAVE) + w] = s;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NV; i += RNTH) {
        double s = lds[i * (RNTH / WAVE)];
        for (int q = 1; q < RNTH / WAVE; q++) {
            const double o = lds[i * (RNTH / WAVE) + q];
            if (i == mx) s = (o > s || o != o) ? o : s;
            else s += o;
        }
        part[(int64_t)i * gridDim.x + blockIdx.x] = s;
    }
}

// out[v] = sum (index mx: maximum) of the `blocks` partials of value v, in a fixed order
__global__ __launch_bounds__(FINISH_WAVES *WAVE) void finish_sums(const double *part, int blocks,
                                                                  int nv, int mx, double *out) {
    const int lane = threadIdx.x & (WAVE - 1);
    for (int v = threadIdx.x / WAVE; v < nv; v += FINISH_WAVES) {
        double s = 0.0;
        for (int b = lane; b < blocks; b += WAVE) {
            const double o = part[(int64_t)v * blocks + b];
            if (v == mx) s = (o > s || o != o) ? o : s;
            else s += o;
        }
        s = v == mx ? wave_max(s) : wave_sum(s);
        if (lane == 0) out[v] = s;
    }
}

// ---- theta: [k] sum_t gamma_k, [K + k*XD + c] sum_t x_c gamma_k over the observed nodes --------
template <typename S, int K, int XD>
__global__ __launch_bounds__(RNTH) void theta_sums(const S *gam, const double *x, InstDesc D,
                                                   double *part) {
    constexpr int NV = K * (1 + XD);
    __shared__ double lds[NV * (RNTH / WAVE)];
    double v[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = 0.0;
    // two nodes at a time (rows start at multiples of 64 elements and reach past T)
    for (int64_t t = 2 * ((int64_t)blockIdx.x * RNTH + threadIdx.x); t < D.T;
         t += 2 * (int64_t)gridDim.x * RNTH) {
        const bool two = t + 1 < D.T;
        bool obs[2] = {true, two};
        if (D.heldout) {
            obs[0] = D.heldout[t] == 0;
            obs[1] = two && D.heldout[t + 1] == 0;
        }
        double xc[XD][2];
#pragma unroll
        for (int c = 0; c < XD; c++) {
            const double2 xv = *reinterpret_cast<const double2 *>(x + D.xoff + c * D.ld + t);
            xc[c][0] = xv.x;
            xc[c][1] = xv.y;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            using V2 = typename std::conditional<sizeof(S) == 8, double2, float2>::type;
            const V2 gv = *reinterpret_cast<const V2 *>(gam + k * D.ld + t);
            const double g[2] = {(double)gv.x, (double)gv.y};
#pragma unroll
            for (int i = 0; i < 2; i++) {
                v[k] += obs[i] ? g[i] : 0.0;
#pragma unroll
                for (int c = 0; c < XD; c++) v[K + k * XD + c] += obs[i] ? xc[c][i] * g[i] : 0.0;
            }
        }
    }
    put_partials<NV>(v, -1, lds, part);
}

static int read_blocks(int64_t nodes) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((nodes + 2 * RNTH - 1) / (2 * RNTH), READ_BLOCKS));
}

template <typename S, int K>
static void launch_theta(hipStream_t s, const S *g, const double *x, const InstDesc &d, double *part,
                         int blocks) {
    if (d.xdim == 1) hipLaunchKernelGGL((theta_sums<S, K, 1>), dim3(blocks), dim3(RNTH), 0, s, g, x, d, part);
    else if (d.xdim == 2) hipLaunchKernelGGL((theta_sums<S, K, 2>), dim3(blocks), dim3(RNTH), 0, s, g, x, d, part);
    else hipLaunchKernelGGL((theta_sums<S, K, 3>), dim3(blocks), dim3(RNTH), 0, s, g, x, d, part);
}

// The theta step (graphh1fem.cpp:374-379: theta_k = <x, gamma_k> / sum(gamma_k), 0 if the sum is
// 0) with its partials at `part` (READ_BLOCKS * K (1 + xdim) doubles).
int theta_from_rows(Engine &e, const void *g, bool f32, const InstDesc &d, const double *x,
                    double *part, double *theta_out) {
    hipStream_t s = (hipStream_t)e.ctx->stream;
    const int blocks = read_blocks(d.T), nv = d.K * (1 + d.xdim);
    switch (d.K) {
#define PASC_TK(KK)                                                                 \
    case KK:                                                                        \
        if (f32) launch_theta<float, KK>(s, (const float *)g, x, d, part, blocks);  \
        else launch_theta<double, KK>(s, (const double *)g, x, d, part, blocks);    \
        break;
        PASC_TK(1) PASC_TK(2) PASC_TK(3) PASC_TK(4) PASC_TK(5) PASC_TK(6) PASC_TK(7) PASC_TK(8)
#undef PASC_TK
        default: return fail(PASC_ERR_ARG, "unsupported K %d", d.K);
    }
    double *tot = reinterpret_cast<double *>(e.h_state);  // pinned; no solve is under way
    hipLaunchKernelGGL(finish_sums, dim3(1), dim3(FINISH_WAVES * WAVE), 0, s, part, blocks, nv, -1, tot);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    for (int k = 0; k < d.K; k++)
        for (int c = 0; c < d.xdim; c++)
            theta_out[k * d.xdim + c] = tot[k] != 0 ? tot[d.K + k * d.xdim + c] / tot[k] : 0.0;
    return PASC_OK;
}

int rows_theta(Engine &e, const void *g, bool f32, const InstDesc &d, const double *x,
               double *theta_out) {
    void *part;
    const int rc = engine_scratch(e, sizeof(double) * READ_BLOCKS * (size_t)d.K * (1 + d.xdim), &part);
    return rc ? rc : theta_from_rows(e, g, f32, d, x, (double *)part, theta_out);
}

// ---- explicit FP64 evaluation: f = 1/2 g'Ag - b'g, ||b||^2 and the KKT residual (max) ----------
// TIME: the 1-D time graph (the neighbour walk without its index arithmetic).
template <typename S, int K, bool TIME>
__global__ __launch_bounds__(RNTH) void eval_sums(const S *gam, const double *x, InstDesc D,
                                                  GraphGeo G, double *part) {
    __shared__ double lds[3 * (RNTH / WAVE)];
    double v[3] = {0.0, 0.0, 0.0};
    for (int64_t t = (int64_t)blockIdx.x * RNTH + threadIdx.x; t < D.T; t += (int64_t)gridDim.x * RNTH) {
        double g0[K], lap[K], q[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            g0[k] = (double)gam[k * D.ld + t];
            lap[k] = 0.0;
            q[k] = 0.0;
        }
        auto add = [&](int64_t n2, double w) {
#pragma unroll
            for (int k = 0; k < K; k++) lap[k] += w * (g0[k] - (double)gam[k * D.ld + n2]);
        };
        if constexpr (TIME) {
            if (t > 0) add(t - 1, 2.0);
            if (t < D.T - 1) add(t + 1, 2.0);
        } else {
            for_neighbours(G, t, add);
        }
        if (D.b64) {
#pragma unroll
            for (int k = 0; k < K; k++) q[k] = -D.b64[k * D.ld + t];
        } else if (!(D.heldout && D.heldout[t])) {
            for (int c = 0; c < D.xdim; c++) {
                const double xc = x[D.xoff + c * D.ld + t];
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const double dx = xc - D.theta[k * D.xdim + c];
                    q[k] += dx * dx;
                }
            }
#pragma unroll
            for (int k = 0; k < K; k++) q[k] *= D.bscale;
        }
        double z[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double g = D.alpha * lap[k] + q[k];
            v[0] += 0.5 * D.alpha * lap[k] * g0[k] + q[k] * g0[k];
            v[1] += q[k] * q[k];
            z[k] = g0[k] - D.s_kkt * g;
        }
        project_simplex<K, double>(z);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double e = fabs(g0[k] - z[k]);
            v[2] = (e > v[2] || e != e) ? e : v[2];
        }
    }
    put_partials<3>(v, 2, lds, part);
}

template <typename S, int K>
static void launch_eval(const Engine &e, const InstDesc &d, const S *g, double *part, int blocks) {
    hipStream_t s = (hipStream_t)e.ctx->stream;
    const double *x = (const double *)e.d_x64;
    if (e.stencil == STENCIL_TIME)
        hipLaunchKernelGGL((eval_sums<S, K, true>), dim3(blocks), dim3(RNTH), 0, s, g, x, d, e.geo, part);
    else
        hipLaunchKernelGGL((eval_sums<S, K, false>), dim3(blocks), dim3(RNTH), 0, s, g, x, d, e.geo, part);
}

int engine_eval_raw(Engine &e, int inst, double *fx, double *kkt, double *nb2) {
    const InstDesc &d = e.h_desc[inst];
    bool f32;
    const void *g = engine_current_gamma(e, inst, &f32);
    const int blocks = read_blocks(d.T);
    void *part;
    int rc = engine_scratch(e, sizeof(double) * 3 * (size_t)READ_BLOCKS, &part);
    if (rc) return rc;
    switch (d.K) {
#define PASC_EK(KK)                                                                        \
    case KK:                                                                               \
        if (f32) launch_eval<float, KK>(e, d, (const float *)g, (double *)part, blocks);   \
        else launch_eval<double, KK>(e, d, (const double *)g, (double *)part, blocks);     \
        break;
        PASC_EK(1) PASC_EK(2) PASC_EK(3) PASC_EK(4) PASC_EK(5) PASC_EK(6) PASC_EK(7) PASC_EK(8)
#undef PASC_EK
        default: return fail(PASC_ERR_ARG, "unsupported K");
    }
    double *tot = reinterpret_cast<double *>(e.h_state);
    hipStream_t s = (hipStream_t)e.ctx->stream;
    hipLaunchKernelGGL(finish_sums, dim3(1), dim3(FINISH_WAVES * WAVE), 0, s, (const double *)part,
                       blocks, 3, 2, tot);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    if (fx) *fx = tot[0];
    if (kkt) *kkt = tot[2];
    if (nb2) *nb2 = tot[1];
    return PASC_OK;
}

// ---- |sum_k theta_k gamma_k - solution|_1: the solution's pieces are read where they are staged,
// each piece leaving one row of partials.  Up to ABS_ONE_WAIT steps this thread copies the solution
// and waits once, for everything.  us of a call, so / staged: T = 1000 18.5 / 31, 40,000 27 / 52, 1e5
// 46 / 71, 2e5 either 90 ----
constexpr int64_t ABS_ONE_WAIT = 160000;
template <typename S>
__global__ __launch_bounds__(RNTH) void abserr_sums(const S *gam, InstDesc D, const double *sol,
                                                    int64_t t0, int64_t n, double *part) {
    __shared__ double lds[RNTH / WAVE];
    double v[1] = {0.0};
    for (int64_t i = (int64_t)blockIdx.x * RNTH + threadIdx.x; i < n; i += (int64_t)gridDim.x * RNTH) {
        double rec = -sol[i];
        for (int k = 0; k < D.K; k++) rec += D.theta[k] * (double)gam[k * D.ld + t0 + i];
        v[0] += fabs(rec);
    }
    put_partials<1>(v, -1, lds, part);
}

int rows_abserr(Engine &e, const void *g, bool f32, const InstDesc &d, const double *solution,
                double *abserr) {
    constexpr int ABS_BLOCKS = 64;
    hipStream_t s = (hipStream_t)e.ctx->stream;
    double *tot = reinterpret_cast<double *>(e.h_state);
    auto finish = [=](const double *part, int rows) {
        hipLaunchKernelGGL(finish_sums, dim3(1), dim3(FINISH_WAVES * WAVE), 0, s, part, rows * ABS_BLOCKS,
                           1, -1, tot);
    };
    auto sums = [=, &d](const void *sol, int64_t t0, int64_t n, double *row) {
        if (f32)
            hipLaunchKernelGGL(abserr_sums<float>, dim3(ABS_BLOCKS), dim3(RNTH), 0, s, (const float *)g, d,
                               (const double *)sol, t0, n, row);
        else
            hipLaunchKernelGGL(abserr_sums<double>, dim3(ABS_BLOCKS), dim3(RNTH), 0, s, (const double *)g,
                               d, (const double *)sol, t0, n, row);
    };
    if (d.T <= ABS_ONE_WAIT) {
        void *part;
        int rc = engine_scratch(e, sizeof(double) * ABS_BLOCKS, &part);
        if (rc == PASC_OK)
            rc = with_input(e.ctx, solution, sizeof(double) * (size_t)d.T, [&](const void *p) {
                sums(p, 0, d.T, (double *)part);
                finish((const double *)part, 1);
            });
        if (rc == PASC_OK) *abserr = tot[0];
        return rc;
    }
    // one row of ABS_BLOCKS partials per piece of the solution
    const int64_t piece = staged_piece(sizeof(double), d.T);
    const int64_t rows = (d.T + piece - 1) / piece;
    void *buf;
    int rc = engine_scratch(e, sizeof(double) * (size_t)(rows * ABS_BLOCKS), &buf);
    if (rc) return rc;
    double *part = (double *)buf;
    rc = staged_transfer(e.ctx, false, const_cast<double *>(solution), sizeof(double), d.T,
                         [=](hipStream_t, int64_t t0, int64_t n, void *p) {
                             sums(p, t0, n, part + t0 / piece * ABS_BLOCKS);
                         });
    if (rc) return rc;
    finish(part, (int)rows);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    *abserr = tot[0];
    return PASC_OK;
}

}  // namespace pasc
