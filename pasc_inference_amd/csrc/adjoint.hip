// Adjoint of the converged gamma step (any graph of the engine, xdim <= 3).
//
// At the minimiser gamma* of  min 1/2 g'Ag - b'g  over the product of simplices, let F be the
// free set {(k,t): gamma_kt > 0} and P the orthogonal projector onto
// {v : v = 0 off F, sum_{k in F_t} v_kt = 0 for every t}.  The KKT conditions P(A gamma - b) = 0
// differentiate to  (P A P) dgamma = -P(dA gamma - db).  For the held-out loss
//   J = sum_{t in M} (x_t - sum_k theta_k gamma_kt)^2
// one CG solve of (P A P) lambda = P dJ/dgamma gives every parameter derivative:
//   dJ/dlog(eps) = -lambda' A gamma                      (A = eps/T A0, so dA/dlog eps = A)
//   dJ/dtheta_k  = dJ/dtheta_k|direct + sum_{t with data} lambda_kt * 2 (x_t - theta_k) / T
// All vectors are FP64, k-major with row stride ld, one thread per time step.  The CG scalars
// (p'APp, r'r, the step and the update factor) are reduced and formed on the device, so an
// iteration needs no host round trip; the host reads the stop flag every CG_POLL iterations.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "device_common.h"
#include "util_kernels.h"

namespace pasc {

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(PASC_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));     \
    } while (0)

constexpr int ANT = 256;
constexpr double FREE_EPS = 1e-12;  // gamma entries at or below this are on the bound

}  // namespace pasc

#include "adjoint_loop.h"

namespace pasc {

struct AdjArgs {
    const double *gam;      // gamma* (k-major, stride ld)
    const double *x;        // data rows [xdim][ld]
    const uint8_t *mask;    // held-out nodes (1 = in the loss)
    const uint8_t *qmask;   // nodes without a data term in the QP (problem's held-out mask)
    uint8_t *freeset;       // [K][ld] 1 = free
    int64_t T, ld;          // T: nodes
    int K, xdim;
    double alpha, bscale;
    double theta[PASC_MAX_K * 3];
    GraphGeo G;
};

constexpr int NTH = PASC_MAX_K * 3;  // theta entries

// Scalars of the CG iteration on the device.  adj_cg_step and adj_cg_rr form them from the
// block partials of the kernel before; the vector kernels read step and b from here and do
// nothing once done is set.
struct CgState {
    double rr, rr0, step, b, tol2;
    int32_t it, maxit, done;
};
constexpr int CG_POLL = 16;  // CG iterations launched between host reads of the stop flag
constexpr int RNT = 1024;    // threads of the one-workgroup partial reductions
constexpr size_t ADJ_KEEP_BYTES = (size_t)1 << 30;

template <int NV>
__device__ inline void block_sum(double (&v)[NV], double *lds, double *out, int block) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = wave_sum(v[i]);
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NV; i++) lds[w * NV + i] = v[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 0; i < NV; i++) {
            double s = 0.0;
            for (int q = 0; q < ANT / WAVE; q++) s += lds[q * NV + i];
            out[(int64_t)block * NV + i] = s;
        }
    }
}

// P applied to the K values of one time step (in place); free flags per k.
template <int K>
__device__ __forceinline__ void project_face(double (&v)[K], const bool (&fr)[K]) {
    int nf = 0;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < K; k++)
        if (fr[k]) { nf++; s += v[k]; }
    const double m = nf > 0 ? s / nf : 0.0;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = (fr[k] && nf > 1) ? v[k] - m : 0.0;
}

// r = P dJ/dgamma; partials: [0] J, [1] r'r, [2 + 3 k + c] direct dJ/dtheta_kc.  (K is a template
// argument here and below so that the values of a step stay in registers.)
template <int K>
__global__ __launch_bounds__(ANT) void adj_init(AdjArgs a, double *r, double *part) {
    constexpr int NV = 2 + 3 * K;
    __shared__ double lds[NV * (ANT / WAVE)];
    const int64_t t = (int64_t)blockIdx.x * ANT + threadIdx.x;
    double v[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = 0.0;
    if (t < a.T) {
        double g[K], dj[K];
        bool fr[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            g[k] = a.gam[k * a.ld + t];
            fr[k] = g[k] > FREE_EPS;
            a.freeset[k * a.ld + t] = fr[k] ? 1 : 0;
            dj[k] = 0.0;
        }
        const bool held = a.mask[t] != 0;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (c >= a.xdim) break;
            double rec = 0.0;
#pragma unroll
            for (int k = 0; k < K; k++) rec += a.theta[k * a.xdim + c] * g[k];
            const double res = held ? a.x[c * a.ld + t] - rec : 0.0;
            v[0] += res * res;
#pragma unroll
            for (int k = 0; k < K; k++) {
                dj[k] += -2.0 * res * a.theta[k * a.xdim + c];
                v[2 + 3 * k + c] = -2.0 * res * g[k];
            }
        }
        project_face<K>(dj, fr);
#pragma unroll
        for (int k = 0; k < K; k++) {
            r[k * a.ld + t] = dj[k];
            v[1] += dj[k] * dj[k];
        }
    }
    block_sum<NV>(v, lds, part, blockIdx.x);
}

// Sum of part[0 .. blocks) in a fixed order (thread i adds blocks i, i + RNT, ..., then the
// workgroup's tree); the result is valid in thread 0.
__device__ inline double reduce_partials(const double *part, int blocks, double *lds) {
    double v = 0.0;
    for (int b = threadIdx.x; b < blocks; b += RNT) v += part[b];
    v = wave_sum(v);
    if ((threadIdx.x & (WAVE - 1)) == 0) lds[threadIdx.x / WAVE] = v;
    __syncthreads();
    double sum = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < RNT / WAVE; i++) sum += lds[i];
    return sum;
}

// after adj_matvec: step = r'r / p'APp, or the stop when p'APp <= 0 (p in the null space of
// P A P, where the system is consistent)
__global__ __launch_bounds__(RNT) void adj_cg_step(const double *part, int blocks, CgState *cs) {
    __shared__ double lds[RNT / WAVE];
    if (cs->done) return;
    const double pq = reduce_partials(part, blocks, lds);
    if (threadIdx.x == 0) {
        if (!(pq > 0.0)) cs->done = 1;
        else cs->step = cs->rr / pq;
    }
}

// after adj_axpy: b = r'r (new) / r'r (old), the iteration counted, and the stop once r'r is
// below tol^2 r'r (initial) or the iterations reach maxit
__global__ __launch_bounds__(RNT) void adj_cg_rr(const double *part, int blocks, CgState *cs) {
    __shared__ double lds[RNT / WAVE];
    if (cs->done) return;
    const double rr_new = reduce_partials(part, blocks, lds);
    if (threadIdx.x == 0) {
        cs->b = rr_new / cs->rr;
        cs->rr = rr_new;
        cs->it += 1;
        if (!(cs->it < cs->maxit && rr_new > cs->tol2 * cs->rr0 && rr_new > 0.0)) cs->done = 1;
    }
}

// The search direction p = r + b pold of this step (b = 0 on the first, where pold = r), written
// to pnew, and q = P A P p (p in range(P)); partial p'q.  pnew and pold are two buffers, since
// the neighbours' pold are read while other workgroups write.
//
// The K components of a neighbour are read together.  On videos the frames before and after are
// then fetched by all eight L2s (40 frames of 100 x 100, K = 3, 20 steps: 1.41 ms, 1.60 with one
// component after the other before, against 1.21 here), unless each XCD has a band of its own
// (xcd_tile).  That pays while a component's three frames of r and p leave room in an L2 of 4 MB:
// ms without / with bands at K = 2 / 4, frames of 30,000 nodes 2.6 / 4.5 against 1.7 / 3.7, of 48,000
// 5.2 / 9.0 against 4.2 / 9.2, of 90,000 2.0 / 3.5 against 2.6 / 4.0.  Images have rows in their
// place: 1024 x 1024, K = 4 2.0 / 1.7, never slower.
constexpr int64_t BAND_FRAME = 40960;
template <int K>
__global__ __launch_bounds__(ANT) void adj_matvec(AdjArgs a, const double *r, const double *pold,
                                                  double *pnew, double *q, double *part,
                                                  const CgState *cs) {
    __shared__ double lds[ANT / WAVE];
    if (cs->done) return;
    const double b = cs->b;
    const bool bands = a.G.R > 1 && (a.G.T == 1 || a.G.R <= BAND_FRAME);
    const int block = bands ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int64_t t = (int64_t)block * ANT + threadIdx.x;
    double v[1] = {0.0};
    if (t < a.T) {
        double w[K], pn[K];
        bool fr[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            pn[k] = r[k * a.ld + t] + b * pold[k * a.ld + t];
            fr[k] = a.freeset[k * a.ld + t] != 0;
            w[k] = 0.0;
        }
        // (A0 p) at the node, p formed at the neighbours too
        for_neighbours(a.G, t, [&](int64_t n2, double wt) {
#pragma unroll
            for (int k = 0; k < K; k++)
                w[k] += wt * (pn[k] - (r[k * a.ld + n2] + b * pold[k * a.ld + n2]));
        });
#pragma unroll
        for (int k = 0; k < K; k++) w[k] *= a.alpha;
        project_face<K>(w, fr);
#pragma unroll
        for (int k = 0; k < K; k++) {
            pnew[k * a.ld + t] = pn[k];
            q[k * a.ld + t] = w[k];
            v[0] += pn[k] * w[k];
        }
    }
    block_sum<1>(v, lds, part, block);
}

// lam += s p; r -= s q with s the step; partial r'r
template <int K>
__global__ __launch_bounds__(ANT) void adj_axpy(AdjArgs a, const CgState *cs, const double *p,
                                                const double *q, double *lam, double *r,
                                                double *part) {
    __shared__ double lds[ANT / WAVE];
    if (cs->done) return;
    const double s = cs->step;
    const int64_t t = (int64_t)blockIdx.x * ANT + threadIdx.x;
    double v[1] = {0.0};
    if (t < a.T) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int64_t i = k * a.ld + t;
            lam[i] += s * p[i];
            const double rn = r[i] - s * q[i];
            r[i] = rn;
            v[0] += rn * rn;
        }
    }
    block_sum<1>(v, lds, part, blockIdx.x);
}

// partials: [0] lambda' A gamma, [1 + 3 k + c] sum_{n with data} lambda_kn 2 (x_nc - theta_kc) bscale
template <int K>
__global__ __launch_bounds__(ANT) void adj_final(AdjArgs a, const double *lam, double *part) {
    constexpr int NV = 1 + 3 * K;
    __shared__ double lds[NV * (ANT / WAVE)];
    const int64_t t = (int64_t)blockIdx.x * ANT + threadIdx.x;
    double v[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = 0.0;
    if (t < a.T) {
        const bool nodata = a.qmask && a.qmask[t] != 0;  // b_kn does not depend on theta there
        double g[K], l[K], lk[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            g[k] = a.gam[k * a.ld + t];
            lk[k] = lam[k * a.ld + t];
            l[k] = 0.0;
        }
        for_neighbours(a.G, t, [&](int64_t n2, double w) {
#pragma unroll
            for (int k = 0; k < K; k++) l[k] += w * (g[k] - a.gam[k * a.ld + n2]);
        });
#pragma unroll
        for (int k = 0; k < K; k++) v[0] += lk[k] * a.alpha * l[k];
        if (!nodata) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (c >= a.xdim) break;
                const double xc = a.x[c * a.ld + t];
#pragma unroll
                for (int k = 0; k < K; k++)
                    v[1 + 3 * k + c] = lk[k] * 2.0 * (xc - a.theta[k * a.xdim + c]) * a.bscale;
            }
        }
    }
    block_sum<NV>(v, lds, part, blockIdx.x);
}

static int sum_partials(hipStream_t s, const double *d_part, int blocks, int nv,
                        std::vector<double> &out) {
    std::vector<double> h((size_t)blocks * nv);
    HIP_TRY(hipMemcpyAsync(h.data(), d_part, sizeof(double) * h.size(), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    out.assign(nv, 0.0);
    for (int b = 0; b < blocks; b++)
        for (int i = 0; i < nv; i++) out[i] += h[(size_t)b * nv + i];
    return PASC_OK;
}

__global__ __launch_bounds__(256) void copy_bytes(const uint8_t *src, uint8_t *dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        dst[i] = src[i];
}

// the caller's mask to the device
static int upload_mask(Engine &e, const uint8_t *mask, uint8_t *dst, int64_t n) {
    return staged_transfer(e.ctx, false, const_cast<uint8_t *>(mask), 1, n,
                           [=](hipStream_t s, int64_t i0, int64_t m, void *p) {
                               const unsigned b = (unsigned)std::min<int64_t>((m + 255) / 256, 1024);
                               hipLaunchKernelGGL(copy_bytes, dim3(b), dim3(256), 0, s,
                                                  (const uint8_t *)p, dst + i0, m);
                           });
}

struct AdjResult {
    double loss, lag;  // J and lambda' A gamma
    double dtheta[PASC_MAX_K * 3];
    int it;
};

// One problem on the 1-D graph whose CG vectors fit on chip: the persistent launch (adjoint_loop.h).
// *ran = false when it does not qualify, the launch is refused or its workgroups lost each other.
template <int K, int CH, int NW>
static bool launch_adj_loop(const AdjLoopArgs &a, int nwg, hipStream_t s) {
    const void *fn = reinterpret_cast<const void *>(adj_loop<K, CH, NW>);
    const size_t lds = (size_t)K * NW * WAVE * CH * sizeof(double);
    AdjLoopArgs args = a;
    void *params[] = {&args};
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess &&
        hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(NW * WAVE), params, (unsigned)lds, s) == hipSuccess)
        return true;
    (void)hipGetLastError();
    return false;
}

template <int K>
static int run_adj_loop(Engine &e, const InstDesc &D, const double *gam, const uint8_t *mask_host,
                        double cg_tol, int cg_maxit, AdjResult &res, bool *ran) {
    *ran = false;
    constexpr int CH = adj_chunk(K);
    const int64_t n_cu = std::max(e.ctx->n_cu, 1);
    auto groups = [&](int steps) { return (D.T + steps - 1) / steps; };
    // 4 waves of half chunks, 8 of half chunks, 8 of whole chunks: the first whose workgroups fit
    const int steps = groups(4 * WAVE * CH / 2) <= n_cu ? 4 * WAVE * CH / 2
                      : groups(8 * WAVE * CH / 2) <= n_cu ? 8 * WAVE * CH / 2 : 8 * WAVE * CH;
    if (groups(steps) > n_cu) return PASC_OK;
    hipStream_t s = (hipStream_t)e.ctx->stream;
    const int nwg = (int)groups(steps);
    const int64_t ew = adj_epoch_words<K>(nwg), ow = adj_open_words<K>(nwg);
    const int64_t cap = std::max<int64_t>(1, LOOP_EXCHANGE_BYTES / (8 * ew));
    const int epochs = (int)std::min<int64_t>(std::max(cg_maxit, 1), std::min<int64_t>(cap, 512));
    // exchange area, r'r, (with more steps than a launch holds) r, p and lambda, the mask
    const int64_t save = cg_maxit > epochs ? 3 * (int64_t)K * D.ld : 0;
    const size_t bytes = sizeof(double) * (size_t)(ow + ew * epochs + 2 + save) + (size_t)D.T;
    void *buf;
    int rc = engine_scratch(e, bytes, &buf);
    if (rc) return rc;
    double *ex = (double *)buf;
    uint8_t *mk = (uint8_t *)(ex + ow + ew * epochs + 2 + save);
    rc = upload_mask(e, mask_host, mk, D.T);
    if (rc) return rc;
    AdjLoopArgs a{};
    a.gam = gam;
    a.x = (const double *)e.d_x64 + D.xoff;
    a.mask = mk;
    a.qmask = D.heldout;
    a.T = D.T;
    a.ld = D.ld;
    a.alpha = D.alpha;
    a.bscale = D.bscale;
    a.tol2 = cg_tol * cg_tol;
    for (int k = 0; k < K; k++) a.theta[k] = D.theta[k];
    a.save_rr = ex + ow + ew * epochs;
    a.save = a.save_rr + 2;
    a.out = (double *)e.h_state;  // pinned; no solve is under way
    a.flags = e.h_poll;
    a.ex = ex;
    a.epochs = epochs;
    a.maxit = cg_maxit;
    for (a.resume = 0;; a.resume = 1) {
        const int64_t words = ow + ew * epochs;
        hipLaunchKernelGGL(fill_u64, dim3((unsigned)std::min<int64_t>((words + 255) / 256, 1024)),
                           dim3(256), 0, s, (uint64_t *)ex, words, PART_EMPTY);
        HIP_TRY(hipGetLastError());
        a.flags[0] = 0;
        a.flags[1] = 0;
        const bool ok = steps == 4 * WAVE * CH / 2   ? launch_adj_loop<K, CH / 2, 4>(a, nwg, s)
                        : steps == 8 * WAVE * CH / 2 ? launch_adj_loop<K, CH / 2, 8>(a, nwg, s)
                                                     : launch_adj_loop<K, CH, 8>(a, nwg, s);
        if (!ok) return PASC_OK;
        HIP_TRY(hipStreamSynchronize(s));
        if (a.flags[1] || e.ctx->take_back) return PASC_OK;  // the workgroups lost each other: nothing of it is used
        if (!a.flags[0]) break;
    }
    res.loss = a.out[0];
    res.lag = a.out[1];
    for (int k = 0; k < K; k++) res.dtheta[k] = a.out[2 + k];
    res.it = a.flags[2];
    *ran = true;
    return PASC_OK;
}

// Any graph, size and number of channels: CG as kernels over vectors in device memory.
template <int K>
static int run_adj_kernels(Engine &e, const InstDesc &D, const uint8_t *mask_host, double cg_tol,
                           int cg_maxit, AdjResult &res) {
    hipStream_t s = (hipStream_t)e.ctx->stream;
    const int64_t T = D.T, ld = D.ld, n = (int64_t)K * ld;
    const int blocks = (int)((T + ANT - 1) / ANT);
    const int par = e.h_parity[0];
    constexpr int NV = 2 + 3 * K;
    // gamma when the state is FP32, lambda, r, q and two buffers of p, the partials, the CG
    // state, the free set and the mask
    const bool f32 = !e.cur64 && e.precision == PASC_FP32_BULK;
    void *mem;
    int rc = engine_scratch(e, sizeof(double) * (size_t)(6 * n + (int64_t)blocks * NV) + 128 +
                                   (size_t)n + (size_t)T, &mem);
    if (rc) return rc;
    double *buf = (double *)mem;
    double *lam = buf + n, *r = buf + 2 * n, *q = buf + 3 * n;
    double *pb[2] = {buf + 4 * n, buf + 5 * n};
    double *part = buf + 6 * n;
    CgState *d_cs = (CgState *)(part + (int64_t)blocks * NV);
    uint8_t *fr = (uint8_t *)d_cs + 128, *mk = fr + n;
    static_assert(sizeof(CgState) <= 128, "the CG state fits its place");
    const double *gam = e.cur64 ? (const double *)e.d_gamma64[par] + D.goff
                                : (const double *)e.d_gamma[par] + D.goff;
    if (f32) {
        gam = buf;
        hipLaunchKernelGGL((convert_kernel<float, double>), dim3((unsigned)((n + 255) / 256)), dim3(256),
                           0, s, (const float *)e.d_gamma[par] + D.goff, buf, n);
        HIP_TRY(hipGetLastError());
    }
    rc = upload_mask(e, mask_host, mk, T);
    if (rc) return rc;
    HIP_TRY(hipMemsetAsync(lam, 0, sizeof(double) * (size_t)n, s));
    AdjArgs a;
    a.gam = gam;
    a.x = (const double *)e.d_x64 + D.xoff;
    a.mask = mk;
    a.qmask = D.heldout;
    a.freeset = fr;
    a.T = T;
    a.ld = ld;
    a.K = K;
    a.xdim = D.xdim;
    a.alpha = D.alpha;
    a.bscale = D.bscale;
    for (int i = 0; i < NTH; i++) a.theta[i] = i < K * D.xdim ? D.theta[i] : 0.0;
    a.G = e.stencil == STENCIL_TIME ? GraphGeo{T, 1, 0, nullptr, nullptr} : e.geo;

    std::vector<double> v;
    hipLaunchKernelGGL(adj_init<K>, dim3(blocks), dim3(ANT), 0, s, a, r, part);
    HIP_TRY(hipGetLastError());
    if ((rc = sum_partials(s, part, blocks, NV, v))) return rc;
    res.loss = v[0];
    for (int k = 0; k < K; k++)
        for (int c = 0; c < D.xdim; c++) res.dtheta[k * D.xdim + c] = v[2 + 3 * k + c];
    HIP_TRY(hipMemcpyAsync(pb[0], r, sizeof(double) * (size_t)n, hipMemcpyDeviceToDevice, s));
    // conjugate gradients on P A P (symmetric positive semi-definite on range(P)), the scalars
    // on the device; the host reads the stop flag every CG_POLL iterations
    CgState h0{};  // the initial state; stays alive until the copies below have completed
    h0.rr = h0.rr0 = v[1];
    h0.tol2 = cg_tol * cg_tol;
    h0.maxit = cg_maxit;
    h0.done = (cg_maxit > 0 && h0.rr > h0.tol2 * h0.rr0 && h0.rr > 0.0) ? 0 : 1;
    HIP_TRY(hipMemcpyAsync(d_cs, &h0, sizeof(CgState), hipMemcpyHostToDevice, s));
    CgState h = h0;
    for (int launched = 0; !h.done && launched <= cg_maxit + CG_POLL; launched += CG_POLL) {
        for (int i = 0; i < CG_POLL; i++) {
            // step launched + i reads p from pb[(launched + i) & 1] and writes the other
            const double *pold = pb[i & 1];
            double *pnew = pb[(i + 1) & 1];
            hipLaunchKernelGGL(adj_matvec<K>, dim3(blocks), dim3(ANT), 0, s, a, r, pold, pnew, q,
                               part, d_cs);
            hipLaunchKernelGGL(adj_cg_step, dim3(1), dim3(RNT), 0, s, part, blocks, d_cs);
            hipLaunchKernelGGL(adj_axpy<K>, dim3(blocks), dim3(ANT), 0, s, a, d_cs, pnew, q, lam, r,
                               part);
            hipLaunchKernelGGL(adj_cg_rr, dim3(1), dim3(RNT), 0, s, part, blocks, d_cs);
        }
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpyAsync(&h, d_cs, sizeof(CgState), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    res.it = h.it;
    hipLaunchKernelGGL(adj_final<K>, dim3(blocks), dim3(ANT), 0, s, a, lam, part);
    HIP_TRY(hipGetLastError());
    if ((rc = sum_partials(s, part, blocks, 1 + 3 * K, v))) return rc;
    res.lag = v[0];
    for (int k = 0; k < K; k++)
        for (int c = 0; c < D.xdim; c++) res.dtheta[k * D.xdim + c] += v[1 + 3 * k + c];
    return PASC_OK;
}

template <int K>
static int run_adj(Engine &e, const InstDesc &D, const uint8_t *mask, double cg_tol, int cg_maxit,
                   AdjResult &res) {
    const bool f32 = !e.cur64 && e.precision == PASC_FP32_BULK;
    if (e.stencil == STENCIL_TIME && D.xdim == 1 && !f32 && !e.profile) {
        const int par = e.h_parity[0];
        const double *gam = (const double *)(e.cur64 ? e.d_gamma64[par] : e.d_gamma[par]) + D.goff;
        bool ran;
        const int rc = run_adj_loop<K>(e, D, gam, mask, cg_tol, cg_maxit, res, &ran);
        if (rc || ran) return rc;
    }
    const int rc = run_adj_kernels<K>(e, D, mask, cg_tol, cg_maxit, res);
    // Six vectors of a large problem (1.4 GB at T = 1e7, K = 3) are not kept with it between its
    // adjoints; up to 1 GiB they are, since a new allocation costs 0.5 - 0.9 ms (3.8 -> 4.4 ms for
    // T = 3e6, K = 3 and 20 steps, 12.3 -> 13.2 for T = 1e7).
    engine_trim_scratch(e, ADJ_KEEP_BYTES);
    return rc;
}

int engine_adjoint(Engine &e, int inst, const uint8_t *mask_host, double cg_tol, int cg_maxit,
                   double *loss, double *dlogeps, double *dtheta, int *cg_it) {
    const InstDesc &D = e.h_desc[inst];
    if (D.b64) return fail(PASC_ERR_ARG, "adjoint: needs the data term");
    AdjResult r{};
    int rc;
    switch (D.K) {
        case 1: rc = run_adj<1>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 2: rc = run_adj<2>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 3: rc = run_adj<3>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 4: rc = run_adj<4>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 5: rc = run_adj<5>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 6: rc = run_adj<6>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 7: rc = run_adj<7>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        case 8: rc = run_adj<8>(e, D, mask_host, cg_tol, cg_maxit, r); break;
        default: rc = fail(PASC_ERR_ARG, "unsupported K");
    }
    if (rc) return rc;
    *loss = r.loss;
    *dlogeps = -r.lag;
    for (int i = 0; i < D.K * D.xdim; i++) dtheta[i] = r.dtheta[i];
    if (cg_it) *cg_it = r.it;
    if (!std::isfinite(*dlogeps)) return fail(PASC_ERR_NUMERIC, "adjoint: non-finite gradient");
    return PASC_OK;
}

}  // namespace pasc
