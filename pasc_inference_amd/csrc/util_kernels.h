// Auxiliary kernels: stand-alone projection and matvec (the kernel-level C-ABI entry points),
// labels, fills and conversions.
#pragma once

#include "device_common.h"

namespace pasc {

// ---- stand-alone projection, K <= 8: one thread per block of K values ----------------------
// layout 0: t-major (block t = x[t*K .. t*K+K-1]);  layout 1: k-major (x[k*ld + t])
template <typename S, typename C, int K>
__global__ __launch_bounds__(256) void project_thread(S *x, int64_t nblocks, int layout,
                                                      int64_t ld) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nblocks) return;
    C y[K];
#pragma unroll
    for (int k = 0; k < K; k++) y[k] = C(layout == 0 ? x[t * K + k] : x[k * ld + t]);
    project_simplex<K, C>(y);
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (layout == 0) x[t * K + k] = S(y[k]);
        else x[k * ld + t] = S(y[k]);
    }
}

// ---- stand-alone projection, large K: one wavefront per block ------------------------------
// Lanes hold the entries k = lane + 64*i.  The threshold is bracketed in [max-1, max) and
// bisected (wave-wide sums), then finished exactly by the support fixed point.
template <typename S>
__global__ __launch_bounds__(256) void project_wave(S *x, int64_t nblocks, int K, int layout,
                                                    int64_t ld) {
    const int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const int lane = threadIdx.x & (WAVE - 1);
    if (b >= nblocks) return;
    auto at = [&](int k) -> int64_t { return layout == 0 ? b * K + k : (int64_t)k * ld + b; };
    double s = 0.0, mx = -1e308;
    int neg = 0;
    for (int k = lane; k < K; k += WAVE) {
        const double v = (double)x[at(k)];
        s += v;
        neg |= v < 0.0;
        mx = v > mx ? v : mx;
    }
    s = wave_sum(s);
    neg = wave_sum_i(neg);
    mx = wave_max(mx);
    if (neg == 0 && s == 1.0) return;
    double lo = mx - 1.0, hi = mx;
    for (int it = 0; it < 24; it++) {
        const double mid = 0.5 * (lo + hi);
        double phi = 0.0;
        for (int k = lane; k < K; k += WAVE) {
            const double v = (double)x[at(k)] - mid;
            phi += v > 0.0 ? v : 0.0;
        }
        phi = wave_sum(phi) - 1.0;
        if (phi >= 0.0) lo = mid; else hi = mid;
    }
    double tau = lo;
    int cnt_prev = -1;
    for (int it = 0; it < K; it++) {
        double sum = 0.0;
        int cnt = 0;
        for (int k = lane; k < K; k += WAVE) {
            const double v = (double)x[at(k)];
            if (v > tau) { sum += v; cnt++; }
        }
        sum = wave_sum(sum);
        cnt = wave_sum_i(cnt);
        if (cnt == cnt_prev || cnt == 0) break;
        cnt_prev = cnt;
        tau = (sum - 1.0) / (double)cnt;
    }
    for (int k = lane; k < K; k += WAVE) {
        const double v = (double)x[at(k)] - tau;
        x[at(k)] = S(v > 0.0 ? v : 0.0);
    }
}

// ---- stand-alone matvec y = alpha*A0*x (k-major rows of stride ld) --------------------------
template <typename S>
__global__ __launch_bounds__(256) void matvec_time(const S *x, S *y, int64_t T, int K,
                                                   int64_t ld, double alpha) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = blockIdx.y;
    if (t >= T || k >= K) return;
    const S *r = x + k * ld;
    double a = 0.0;
    if (t > 0) a += 2.0 * ((double)r[t] - (double)r[t - 1]);
    if (t < T - 1) a += 2.0 * ((double)r[t] - (double)r[t + 1]);
    y[k * ld + t] = S(alpha * a);
}

template <typename S>
__global__ __launch_bounds__(256) void matvec_graph(const S *x, S *y, GraphGeo G, int K,
                                                    int64_t ld, double alpha) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = blockIdx.y;
    if (n >= G.T * G.R || k >= K) return;
    const S *v = x + k * ld;
    const double c = (double)v[n];
    double a = 0.0;
    for_neighbours(G, n, [&](int64_t n2, double w) { a += w * (c - (double)v[n2]); });
    y[k * ld + n] = S(alpha * a);
}

// ---- labels (argmax over k, lowest k on ties) -------------------------------------------------
template <typename S>
__global__ __launch_bounds__(256) void labels_kernel(const S *gam, int64_t n, int64_t ld, int K,
                                                     int32_t *lab) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    int best = 0;
    double bv = (double)gam[t];
    for (int k = 1; k < K; k++) {
        const double v = (double)gam[k * ld + t];
        if (v > bv) { bv = v; best = k; }
    }
    lab[t] = best;
}

// ---- element-wise conversion (FP32 state -> FP64 polish state) ------------------------------
template <typename A, typename B>
__global__ __launch_bounds__(256) void convert_kernel(const A *src, B *dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = B(src[i]);
}

// ---- fill of 64-bit words (the PART_EMPTY marks of the fused step's partial sums) ----------
static __global__ __launch_bounds__(256) void fill_u64(uint64_t *p, int64_t n, uint64_t v) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        p[i] = v;
}

// ---- a single problem's descriptor and, with put_state, its initial state, handed over in kernel
// arguments; the persistent loop's exchange area (n words) is marked empty by the same launch ----
static __global__ __launch_bounds__(256) void prepare_single(InstDesc *desc, InstDesc d,
                                                             InstState *state, InstState st,
                                                             int put_state, uint64_t *ex, int64_t n) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *desc = d;
        if (put_state) *state = st;
    }
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        ex[i] = PART_EMPTY;
}

// ---- last gamma row ----------------------------------------------------------------------------
// The fused 1-D pass and the graph kernels store K - 1 rows of each iterate (the last is 1 - the
// sum of the others, clamped at 0).  At the end of a phase this writes the full last row of every instance's
// current iterate, with the pass's own arithmetic, so that the row equals the value the pass
// used.  Instances that ran no pass in the phase (first still set) keep their rows.  grid.y
// strides over the instances, grid.x over the steps (the nodes, for a graph).
template <typename S>
__global__ __launch_bounds__(256) void complete_last_row(const InstDesc *desc,
                                                         const InstState *state, int n_inst,
                                                         S *g0, S *g1) {
    for (int i = blockIdx.y; i < n_inst; i += gridDim.y) {
        const InstDesc &D = desc[i];
        const int K = D.K;
        if (K < 2 || state[i].first) continue;
        S *g = (state[i].parity ? g1 : g0) + D.goff;
        for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < D.T;
             t += (int64_t)gridDim.x * 256) {
            S r = S(1);
            for (int k = 0; k < K - 1; k++) r -= g[k * D.ld + t];
            g[(K - 1) * D.ld + t] = r > S(0) ? r : S(0);
        }
    }
}

}  // namespace pasc
