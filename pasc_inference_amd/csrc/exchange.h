// Building blocks of the persistent kernels: sums over a wave in registers, and the exchange of a
// few values between workgroups that run at the same time (loop_kernels.h, adjoint_loop.h).
#pragma once

#include "device_common.h"

namespace pasc {

// Re-reads (~1 us each) before a value counts as lost.  A constant: as a kernel argument it took a
// scalar register that the adjoint's loop does not have (0.8 % of its call, 1.7 % kept in one).
constexpr int LOOP_SPIN_LIMIT = 1 << 22;
constexpr size_t LOOP_LDS_BYTES = 159 * 1024;      // dynamic LDS (160 KiB less the static part)
constexpr int64_t LOOP_EXCHANGE_BYTES = 16 << 20;  // exchange area of a launch at most

// The exchange area holds each exchanged sum as one row over the workgroups (a wave reads 64
// workgroups' values as 512 contiguous bytes).
__host__ __device__ constexpr int slot_stride(int nwg) { return (nwg + 15) / 16 * 16; }

// Every workgroup publishes its sums SUM_COPIES times and reads one copy: the workgroups that meet
// at one cache line, where they queue, are as many times fewer.  us per iteration with 1 / 2 / 4 / 8
// copies: 250 x 150 image 6.4 / 5.6 / 5.4 / 5.3, 60 frames of 64 x 48 11.6 / 11.0 / 10.7 / 10.6,
// 1024 x 1024 13.2 / 12.6 / 12.4 / 12.4, series of 2.5e5 steps 5.6 / 5.5 / 5.5 / 5.8.
constexpr int SUM_COPIES = 4;

// ---- wave-wide sums by lane swaps and DPP (VALU moves; no LDS round trips) -------------------
template <int CTRL>
__device__ __forceinline__ double dpp_from(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)(unsigned)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double join_words(unsigned lo, unsigned hi) {
    return __longlong_as_double(((long long)hi << 32) | (long long)lo);
}
// a's upper 32 lanes <-> b's lower 32 lanes (v_permlane32_swap), and a's odd rows of 16 lanes <->
// b's even rows (v_permlane16_swap): after either, a + b holds a's pairwise sums in one half of
// the lanes and b's in the other, so two values are folded by two swaps and one add
__device__ __forceinline__ double fold32(double a, double b) {
    const long long u = __double_as_longlong(a), w = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)w, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(w >> 32), false, false);
    return join_words(lo[0], hi[0]) + join_words(lo[1], hi[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
    const long long u = __double_as_longlong(a), w = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)w, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(w >> 32), false, false);
    return join_words(lo[0], hi[0]) + join_words(lo[1], hi[1]);
}
constexpr int DPP_ROR = 0x120;          // + n: rotate within a row of 16 lanes
constexpr int DPP_XOR1 = 0xB1;          // quad_perm 1,0,3,2
constexpr int DPP_XOR2 = 0x4E;          // quad_perm 2,3,0,1
constexpr int DPP_HALF_MIRROR = 0x141;  // lane i <- lane 7 - i of its half row
// sums of four values over the wave: every lane of row 0 / 1 / 2 / 3 (16 lanes each) ends with
// the sum of a / c / b / d
__device__ __forceinline__ double wave_sum4(double a, double b, double c, double d) {
    double v = fold16(fold32(a, b), fold32(c, d));
    v += dpp_from<DPP_ROR + 8>(v);
    v += dpp_from<DPP_ROR + 4>(v);
    v += dpp_from<DPP_ROR + 2>(v);
    v += dpp_from<DPP_ROR + 1>(v);
    return v;
}
constexpr int ROW_A = 0, ROW_B = 32, ROW_C = 16, ROW_D = 48;  // a lane of each sum
__device__ __forceinline__ double nan_max(double a, double b) { return (b > a || b != b) ? b : a; }
// maximum over the wave (a NaN wins), in every lane
__device__ __forceinline__ double wave_max_all(double v) {
    v = nan_max(v, dpp_from<DPP_ROR + 8>(v));
    v = nan_max(v, dpp_from<DPP_ROR + 4>(v));
    v = nan_max(v, dpp_from<DPP_ROR + 2>(v));
    v = nan_max(v, dpp_from<DPP_ROR + 1>(v));
    return nan_max(nan_max(lane_value(v, 0), lane_value(v, 16)),
                   nan_max(lane_value(v, 32), lane_value(v, 48)));
}

// sum over the wave, in every lane
__device__ __forceinline__ double wave_sum_all(double v) {
    v += dpp_from<DPP_ROR + 8>(v);
    v += dpp_from<DPP_ROR + 4>(v);
    v += dpp_from<DPP_ROR + 2>(v);
    v += dpp_from<DPP_ROR + 1>(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

__device__ __forceinline__ bool published(double v) {
    return __builtin_bit_cast(uint64_t, v) != PART_EMPTY;
}

// One value that another workgroup publishes at p; *lost is set when it does not come.
__device__ __forceinline__ double await_value(const double *p, int32_t *lost) {
    double v = load_coherent(p);
    for (int n = 0; !published(v) && n < LOOP_SPIN_LIMIT; n++) v = load_coherent(p);
    if (!published(v)) *lost = 1;
    return v;
}

// Sum of the n workgroups' values row[0 .. n), in index order per lane; called by a whole wave.
// All values of a lane are re-read together until the last one is there.
__device__ __forceinline__ double await_sum(const double *row, int n, int lane, int32_t *lost) {
    double s = 0.0;
    for (int j0 = lane; j0 < n; j0 += 4 * WAVE) {
        double w[4];
        bool all;
        int spins = 0;
        do {
            all = true;
#pragma unroll
            for (int b = 0; b < 4; b++) w[b] = j0 + b * WAVE < n ? load_coherent(row + j0 + b * WAVE) : 0.0;
#pragma unroll
            for (int b = 0; b < 4; b++) all = all && published(w[b]);
        } while (!all && ++spins < LOOP_SPIN_LIMIT);
        if (!all) *lost = 1;
#pragma unroll
        for (int b = 0; b < 4; b++) s += w[b];
    }
    return wave_sum_all(s);
}

}  // namespace pasc
