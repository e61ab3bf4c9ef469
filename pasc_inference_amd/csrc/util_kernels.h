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

// ---- stand-alone matvec y = alpha*A0*x (k-major rows of stride ld) --------------------------
// Time graph: a wave covers MV_SEG segments of 64 consecutive steps, all loaded before any is used;
// the neighbours come from the adjacent lanes and segments, so a step is loaded once per wave
// (rows of any stride and alignment: 8- or 4-byte loads).  One step a thread with three loads
// each took 23.8 us for 2 million steps of 3 rows in FP64 (96 MB).
constexpr int MV_SEG = 4;
template <typename S>
__global__ __launch_bounds__(256) void matvec_time(const S *x, S *y, int64_t T, int K,
                                                   int64_t ld, double alpha) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t t0 = (((int64_t)blockIdx.x * 256 + threadIdx.x) / WAVE) * (WAVE * MV_SEG);
    const int k = blockIdx.y;
    if (t0 >= T) return;
    const S *r = x + k * ld;
    double v[MV_SEG], before = 0.0, after = 0.0;
#pragma unroll
    for (int j = 0; j < MV_SEG; j++) {
        const int64_t t = t0 + j * WAVE + lane;
        v[j] = t < T ? (double)r[t] : 0.0;
    }
    if (lane == 0 && t0 > 0) before = (double)r[t0 - 1];
    if (lane == WAVE - 1 && t0 + WAVE * MV_SEG < T) after = (double)r[t0 + WAVE * MV_SEG];
#pragma unroll
    for (int j = 0; j < MV_SEG; j++) {
        const int64_t t = t0 + j * WAVE + lane;
        // the lane before and after, at the segment's ends the neighbouring segment's end
        double left = dpp_shift<DPP_WAVE_SHR1>(v[j]), right = dpp_shift<DPP_WAVE_SHL1>(v[j]);
        const double lastl = j > 0 ? lane_value(v[j > 0 ? j - 1 : 0], WAVE - 1) : before;
        const double firstr = j < MV_SEG - 1 ? lane_value(v[j < MV_SEG - 1 ? j + 1 : j], 0) : after;
        left = lane == 0 ? lastl : left;
        right = lane == WAVE - 1 ? firstr : right;
        double a = 0.0;
        if (t > 0) a += 2.0 * (v[j] - left);
        if (t < T - 1) a += 2.0 * (v[j] - right);
        if (t < T) y[k * ld + t] = S(alpha * a);
    }
}

// Image (T = 1 on the 4-neighbour grid): a thread walks MV_ROWS rows of its column with the rows
// above and below in registers; the sum's order (up, left, right, down) is the general walk's.
constexpr int MV_ROWS = 8;
template <typename S>
__global__ __launch_bounds__(256) void matvec_image(const S *x, S *y, int32_t W, int32_t H,
                                                    int64_t ld, double alpha) {
    const int col = blockIdx.x * 64 + (threadIdx.x & 63);
    const int r0 = (blockIdx.y * 4 + threadIdx.x / 64) * MV_ROWS;
    if (col >= W || r0 >= H) return;
    const S *v = x + blockIdx.z * ld;
    S *o = y + blockIdx.z * ld;
    const int64_t n0 = (int64_t)r0 * W + col;
    double up = r0 > 0 ? (double)v[n0 - W] : 0.0, c = (double)v[n0];
#pragma unroll
    for (int j = 0; j < MV_ROWS; j++) {
        const int r = r0 + j;
        if (r >= H) break;
        const int64_t n = n0 + (int64_t)j * W;
        const double dn = r + 1 < H ? (double)v[n + W] : 0.0;
        double a = 0.0;
        if (r > 0) a += c - up;
        if (col > 0) a += c - (double)v[n - 1];
        if (col < W - 1) a += c - (double)v[n + 1];
        if (r + 1 < H) a += c - dn;
        o[n] = S(alpha * a);
        up = c;
        c = dn;
    }
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
