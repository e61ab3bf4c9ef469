// Stand-alone simplex projection of blocks with more than 8 values (the kernel-level entry point;
// up to 8 values a thread projects a block with project_simplex).
//
// Every block is read once, held in registers through the search and written once, where its size
// allows; the lanes are laid out so that consecutive lanes touch consecutive memory:
//   * t-major (the K values of a block adjacent): 16 lanes a block up to K = 128, the sums by
//     rotations within a row of 16 lanes; a whole wave a block up to K = 1024;
//   * k-major (blocks adjacent): with many blocks one lane a block, its K values in registers up
//     to K = 64, else re-read from memory in each sweep; with few (the rule at
//     launch_project_many) a whole wave a block as above.
// One wave a block with its values re-read in ~30 sweeps (24 of them bisections) and, k-major, one
// cache line a lane, took 2340 us for 667,000 blocks of 12 doubles, 570 / 740 us (t- / k-major) for
// 160,000 of 50 and 165 / 2060 us for 27,000 of 300; now 55 / 30, 30 / 32 and 31 / 105 us (64 MB
// read and written: 23 us at the copy rate).
// The threshold is the fixed point of tau = (sum_{y > tau} y - 1) / |{y > tau}| from the lower
// bound max(y) - 1: the support only shrinks, so a repeated count ends the search.  All sums are
// FP64.  A block that is feasible already (no negative value, sum exactly 1) is left alone.
#pragma once

#include "exchange.h"

namespace pasc {

// Sums over a group of lanes holding one block; every lane of the group gets the result.
struct Lanes1 {  // one lane
    __device__ static double sum(double v) { return v; }
    __device__ static double max(double v) { return v; }
};
struct Lanes16 {
    __device__ static double sum(double v) {
        v += dpp_from<DPP_ROR + 8>(v);
        v += dpp_from<DPP_ROR + 4>(v);
        v += dpp_from<DPP_ROR + 2>(v);
        return v + dpp_from<DPP_ROR + 1>(v);
    }
    __device__ static double max(double v) {
        v = cmax(v, dpp_from<DPP_ROR + 8>(v));
        v = cmax(v, dpp_from<DPP_ROR + 4>(v));
        v = cmax(v, dpp_from<DPP_ROR + 2>(v));
        return cmax(v, dpp_from<DPP_ROR + 1>(v));
    }
};
struct Lanes64 {
    __device__ static double sum(double v) { return wave_sum_all(v); }
    __device__ static double max(double v) {
        v = Lanes16::max(v);
        return cmax(cmax(lane_value(v, 0), lane_value(v, 16)), cmax(lane_value(v, 32), lane_value(v, 48)));
    }
};

constexpr double PROJ_LOW = -1e308;  // what a place without a value holds: never above a threshold

// Threshold of a block whose values fn(i), i < nv <= n, each lane of the group enumerates; false:
// the block is feasible.  Places from nv on hold PROJ_LOW.  They are told by their index: an
// entry of the block may have that value, and is negative like any other.  In the search their
// values, and NaN, compare false.
template <typename G, typename F>
__device__ __forceinline__ bool block_tau(int n, int nv, int K, F fn, double &tau) {
    double s = 0.0, mx = PROJ_LOW, neg = 0.0;
    for (int i = 0; i < n; i++) {
        const double v = fn(i);
        if (i >= nv) continue;
        s += v;
        neg += v < 0.0 ? 1.0 : 0.0;
        mx = v > mx ? v : mx;
    }
    s = G::sum(s);
    neg = G::sum(neg);
    mx = G::max(mx);
    tau = mx - 1.0;
    bool go = !(neg == 0.0 && s == 1.0);
    const bool project = go;
    double last = -1.0;
    for (int it = 0; it < K; it++) {
        double sum = 0.0, cnt = 0.0;
        for (int i = 0; i < n; i++) {
            const double v = fn(i);
            const bool in = v > tau;
            sum += in ? v : 0.0;
            cnt += in ? 1.0 : 0.0;
        }
        sum = G::sum(sum);
        cnt = G::sum(cnt);
        // the groups of a wave end their searches at different sweeps
        go = go && cnt != last && cnt != 0.0;
        if (go) tau = (sum - 1.0) / cnt;
        last = cnt;
        if (__ballot(go) == 0) break;
    }
    return project;
}

// LANES lanes a block, R values a lane (K <= LANES * R); value k of block b at x[b * bs + k * ks]
template <typename S, typename G, int LANES, int R>
__global__ __launch_bounds__(256) void project_group(S *x, int64_t nblocks, int K, int64_t bs,
                                                     int64_t ks) {
    const int64_t b = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LANES;
    const int l = threadIdx.x & (LANES - 1);
    const bool in = b < nblocks;  // (every lane stays for the wave's ballots)
    S *xb = x + (in ? b : 0) * bs;
    const int nv = in ? (K - l + LANES - 1) / LANES : 0;
    double y[R];
#pragma unroll
    for (int i = 0; i < R; i++) y[i] = i < nv ? (double)xb[(l + i * LANES) * ks] : PROJ_LOW;
    double tau;
    const bool project = block_tau<G>(R, nv, K, [&](int i) { return y[i]; }, tau);
    if (!in || !project) return;
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int k = l + i * LANES;
        const double v = y[i] - tau;
        if (k < K) xb[k * ks] = S(v > 0.0 ? v : 0.0);
    }
}

// one lane a block, k-major rows of stride ld, K <= KM values in registers
template <typename S, int KM>
__global__ __launch_bounds__(256) void project_lane(S *x, int64_t nblocks, int K, int64_t ld) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool in = b < nblocks;
    S *xb = x + (in ? b : 0);
    double y[KM];
#pragma unroll
    for (int k = 0; k < KM; k++) y[k] = in && k < K ? (double)xb[k * ld] : PROJ_LOW;
    double tau;
    const bool project = block_tau<Lanes1>(KM, in ? K : 0, K, [&](int i) { return y[i]; }, tau);
    if (!in || !project) return;
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const double v = y[k] - tau;
        if (k < K) xb[k * ld] = S(v > 0.0 ? v : 0.0);
    }
}

// The same with the values left in memory (K beyond what the registers hold).
template <typename S>
__global__ __launch_bounds__(256) void project_lane_mem(S *x, int64_t nblocks, int K, int64_t ld) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool in = b < nblocks;
    S *xb = x + (in ? b : 0);
    double tau;
    const bool project =
        block_tau<Lanes1>(K, in ? K : 0, K, [&](int k) { return in ? (double)xb[k * ld] : PROJ_LOW; }, tau);
    if (!in || !project) return;
    for (int k = 0; k < K; k++) {
        const double v = (double)xb[k * ld] - tau;
        xb[k * ld] = S(v > 0.0 ? v : 0.0);
    }
}
template <typename S>
__global__ __launch_bounds__(256) void project_wave_mem(S *x, int64_t nblocks, int K, int64_t bs,
                                                        int64_t ks) {
    const int64_t b = ((int64_t)blockIdx.x * 256 + threadIdx.x) / WAVE;
    const int lane = threadIdx.x & (WAVE - 1);
    if (b >= nblocks) return;
    S *xb = x + b * bs;
    double tau;
    const bool project = block_tau<Lanes64>(
        (K + WAVE - 1) / WAVE, (K - lane + WAVE - 1) / WAVE, K,
        [&](int i) {
            const int k = lane + i * WAVE;
            return k < K ? (double)xb[k * ks] : PROJ_LOW;
        },
        tau);
    if (!project) return;
    for (int k = lane; k < K; k += WAVE) {
        const double v = (double)xb[k * ks] - tau;
        xb[k * ks] = S(v > 0.0 ? v : 0.0);
    }
}

// Launches the kernel for K > 8 values a block.
//
// k-major: a wave a block reads a cache line a lane and value, a lane a block one line for all
// lanes but has K values in a row to wait for, so its time hardly depends on the number of blocks
// until the chip is full.  us, lane / wave a block: 1024 blocks of 33 16.6 / 6.2, of 300 425 / 12,
// of 2000 3380 / 164; 8192 of 33 17.4 / 13.3, of 64 19.6 / 16.8; 12,288 of 33 17.9 / 17.9, of 64
// 19.8 / 21; 131,072 of 65 197 / 122, of 300 1560 / 610; 262,144 of 65 224 / 263; 16,384 of
// 2000 7500 / 4780, 32,768 10,510 / 10,340.
template <typename S>
static void launch_project_many(S *x, int64_t nb, int K, bool tmajor, int64_t ld, hipStream_t s) {
    auto blocks = [&](int lanes) { return dim3((unsigned)((nb * lanes + 255) / 256)); };
    const dim3 t(256);
    const int64_t bs = tmajor ? K : 1, ks = tmajor ? 1 : ld;
#define PASC_GROUP(G, LANES, R) \
    hipLaunchKernelGGL((project_group<S, G, LANES, R>), blocks(LANES), t, 0, s, x, nb, K, bs, ks)
    if (tmajor && K <= 128) {
        if (K <= 16) PASC_GROUP(Lanes16, 16, 1);
        else if (K <= 32) PASC_GROUP(Lanes16, 16, 2);
        else if (K <= 64) PASC_GROUP(Lanes16, 16, 4);
        else PASC_GROUP(Lanes16, 16, 8);
    } else if (tmajor || (K > 32 && nb <= (K <= 64 ? 8192 : K <= 1024 ? 131072 : 16384))) {
        if (K <= 64) PASC_GROUP(Lanes64, 64, 1);
        else if (K <= 128) PASC_GROUP(Lanes64, 64, 2);
        else if (K <= 256) PASC_GROUP(Lanes64, 64, 4);
        else if (K <= 512) PASC_GROUP(Lanes64, 64, 8);
        else if (K <= 1024) PASC_GROUP(Lanes64, 64, 16);
        else hipLaunchKernelGGL((project_wave_mem<S>), blocks(64), t, 0, s, x, nb, K, bs, ks);
    } else {
        if (K <= 16) hipLaunchKernelGGL((project_lane<S, 16>), blocks(1), t, 0, s, x, nb, K, ld);
        else if (K <= 32) hipLaunchKernelGGL((project_lane<S, 32>), blocks(1), t, 0, s, x, nb, K, ld);
        else if (K <= 64) hipLaunchKernelGGL((project_lane<S, 64>), blocks(1), t, 0, s, x, nb, K, ld);
        else hipLaunchKernelGGL((project_lane_mem<S>), blocks(1), t, 0, s, x, nb, K, ld);
    }
#undef PASC_GROUP
}

}  // namespace pasc
