// Persistent SPG loop for one 1-D problem whose iterate and data fit in the LDS of the device: one
// launch runs many iterations, with the iterate on chip between them.
//
// The tiled pass (spg_pass_1d) is one launch per iteration.  At T = 1e4 .. 1e6 its bytes take a
// fraction of its time: launch, ramp, the load - exchange - compute - store chain of a tile and
// the hand-over to the last workgroup made 12.4 us (T = 1e4, K = 2) to 25 us (T = 1e6, K = 3) a
// pass, and 27 - 36 us an iteration with a host poll in between.
//
// Here workgroup w owns `tpw` consecutive one-wave tiles (the tiles of the 64-thread pass: 64
// lanes x CH steps, HT halo lanes a side) and keeps their K - 1 gamma rows and data row in LDS.
// An iteration is
//   * every wave: the three levels of its tiles (pass_levels, the tiled pass's arithmetic), the
//     new rows back to LDS, the tiles' outer 3 steps to the LDS edge buffer of the neighbouring
//     tiles and, at the workgroup's two ends, to the exchange area in device memory;
//   * wave 0: the workgroup's five sums to its slot of the exchange area, then all workgroups'
//     slots read back and summed in slot order.  Every workgroup does this for itself, so that
//     one device-memory latency separates two iterations (2.0 - 2.7 us for 11 - 256 workgroups)
//     instead of the four of a counter, a reader, a step and a broadcast;
//   * wave 0: the SPG step on those sums (the same bits in every workgroup); wave 1: the
//     neighbouring workgroups' edge steps from the exchange area.
// Every location of the exchange area is written once per launch: it starts as PART_EMPTY and a
// reader re-reads it until the value is there (settle_published), so no two locations need an
// order between them, and nothing has to be reset inside the launch.  The workgroups must run
// at the same time: the launch is cooperative (one workgroup per CU), which the runtime grants
// only if they all fit.  Waits are bounded: where a value does not come (work of another stream or
// process keeps a workgroup off the chip) the launch is taken back and the phase goes on with the
// tiled passes from where the launch began.  The launch therefore leaves its results in the
// buffer it does not start from.
#pragma once

#include "exchange.h"
#include "spg_kernels.h"

namespace pasc {


constexpr int LOOP_WAVES_MIN = 4;         // waves per workgroup: one per SIMD of the CU,
constexpr int LOOP_WAVES_MAX = 8;         // or two when a workgroup has more than 4 tiles
constexpr int LOOP_EPOCHS_MAX = 512;                 // iterations per launch at most

struct LoopArgs {
    PassArgs p;          // buffers, descriptor, state and step of the problem (grp, part and the
                         // counters are not used)
    double *ex;          // exchange area: `epochs` x (sums of nwg workgroups, then nwg x 2 edges)
    InstState *out;      // pinned host copy of the final state
    int32_t *flags;      // pinned host words: [0] the instance is still active, [1] a wait ran out
    int32_t ntiles;      // one-wave tiles of the series
    int32_t tpw;         // tiles per workgroup
    int32_t epochs;      // iterations of this launch at most
    int32_t kkt_last;    // 1: the KKT residual is evaluated once, for the iterate that stopped
                         // (the area holds one more epoch for it)
};

// Steps per lane.  FP64: 4, or 2 where 4 steps of K values in four arrays would spill (K >= 5)
// and where the series then still has a wave on its own SIMD for every tile (a tile's time, the
// latency of its chains, halves; see loop_plan).  FP32 keeps 4, the chunk of the default tiled
// pass: a thread's FP32 sums cover its chunk, so the chunk fixes their rounding.
constexpr bool loop_has_chunk(bool f64, int K, int ch) {
    return f64 ? ch == 2 || (ch == 4 && K <= 4) : ch == 4;
}

__host__ __device__ constexpr int64_t sum_words(int nwg) {
    return (int64_t)SUM_COPIES * NPART * slot_stride(nwg);
}

// Layout of a workgroup's dynamic LDS and of the exchange area, used on both sides.
template <typename S, int K, int CH>
struct LoopShape {
    static constexpr int HT = halo_threads<CH>();
    static constexpr int TILE = tile_steps<WAVE, CH>();
    static constexpr int KS = stored_rows<K>();
    static constexpr int HE = HT * CH;            // steps of an edge (>= 3)
    static constexpr int ROW = WAVE * CH;         // elements of a tile's row in LDS
    static constexpr int EDGE = KS * HE;          // elements of one side of a tile
    static constexpr size_t TILE_BYTES = (size_t)(KS + 1) * ROW * sizeof(S);
    static constexpr size_t EDGE_BYTES = (size_t)2 * 2 * EDGE * sizeof(S);  // two parities, sides
    static constexpr size_t lds_bytes(int tpw) {
        return (size_t)tpw * (TILE_BYTES + WAVE) + (size_t)(tpw + 2) * EDGE_BYTES;
    }
    static constexpr int64_t epoch_words(int nwg) {
        return sum_words(nwg) + (int64_t)nwg * 2 * EDGE;
    }
};

// The scalar fields of InstState, in registers of wave 0 (the same in every lane).
struct LoopState {
    double f, f_prev, dd_prev, dAd_prev, dd, dAd, gd, alpha_dir, alpha_apply, beta_apply, kkt,
        best_kkt, normb;
    int32_t fs_last, it, first, active, reason, status, stall, parity, it_base;
};

// The window of f with value i in lane i.  `rest` is the maximum without the entry that the next
// push replaces: it does not need the new f, so it is formed while the sums are awaited.
struct LaneWindow {
    double &v;
    double rest;
    int lane;
    double top;
    __device__ void fill(double f, int m) {
        v = lane < m ? f : -__builtin_huge_val();
        top = f;
    }
    __device__ void push(double f, int at) {
        v = lane == at ? f : v;
        top = f > rest ? f : rest;
    }
    __device__ double max(int) const { return top; }
};

__device__ __forceinline__ void loop_load_state(const InstState &g, int m, int lane, LoopState &st,
                                                double &window) {
    st.f = g.f; st.f_prev = g.f_prev; st.dd_prev = g.dd_prev; st.dAd_prev = g.dAd_prev;
    st.dd = g.dd; st.dAd = g.dAd; st.gd = g.gd; st.alpha_dir = g.alpha_dir;
    st.alpha_apply = g.alpha_apply; st.beta_apply = g.beta_apply; st.kkt = g.kkt;
    st.best_kkt = g.best_kkt; st.normb = g.normb; st.fs_last = g.fs_last; st.it = g.it;
    st.first = g.first; st.active = g.active; st.reason = g.reason; st.status = g.status;
    st.stall = g.stall; st.parity = g.parity; st.it_base = g.it_base;
    window = lane < m ? g.fs[lane] : -__builtin_huge_val();
}

__device__ __forceinline__ void loop_put_state(InstState &g, int m, int lane, const LoopState &st,
                                               double window) {
    if (lane < m) g.fs[lane] = window;
    if (lane != 0) return;
    g.f = st.f; g.f_prev = st.f_prev; g.dd_prev = st.dd_prev; g.dAd_prev = st.dAd_prev;
    g.dd = st.dd; g.dAd = st.dAd; g.gd = st.gd; g.alpha_dir = st.alpha_dir;
    g.alpha_apply = st.alpha_apply; g.beta_apply = st.beta_apply; g.kkt = st.kkt;
    g.best_kkt = st.best_kkt; g.normb = st.normb; g.fs_last = st.fs_last; g.it = st.it;
    g.first = st.first; g.active = st.active; g.reason = st.reason; g.status = st.status;
    g.stall = st.stall; g.parity = st.parity; g.it_base = st.it_base;
}

// LDS of the exchange: the waves' sums, and what the waves need of the step (written by wave 0).
struct LoopShared {
    double red[NPART][8];  // [sum][wave]; waves from NW on stay 0
    double a_apply, b_apply, a_dir;
    int32_t it, active;
    int32_t parity;  // the buffer the launch ends in: the one it does not start from
};

// A wave's share of the iteration's sums dd, (sum of the edge terms), dd + off, f, residual: four
// by lane folds, the residual (a maximum) where it is wanted.
template <int NW>
__device__ __forceinline__ void loop_sums(LoopShared &sh, double (&acc)[NPART], bool want_kkt,
                                          int lane, int wave) {
    const double sums = wave_sum4(acc[0], acc[1], acc[2], acc[3]);
    if (want_kkt) acc[4] = wave_max_all(acc[4]);
    if ((lane & 15) == 0)
        sh.red[lane == ROW_A ? 0 : lane == ROW_B ? 1 : lane == ROW_C ? 2 : 3][wave] = sums;
    if (lane == 1) sh.red[4][wave] = acc[4];
}

// Wave 0, after a barrier: the workgroup's sums to its place in the exchange area's rows, every
// workgroup's sums added up, and the SPG step on them (the same bits in every workgroup).
// edge_scale: d'Ad = edge_scale * (sum of the edge terms).
__device__ __forceinline__ void loop_step(LoopShared &sh, bool want_kkt, double edge_scale,
                                          double a_dir, double sample_eps, double *ex, int slot_ld,
                                          int nwg, int wg, int lane, LoopState &st, double &window,
                                          const StepParams &sp, int32_t *flags) {
    // lane 8 q + w holds wave w's value q; three exchanges sum over w
    double v0 = lane < 8 * NPART ? sh.red[lane >> 3][lane & 7] : 0.0, v1 = v0;
    v0 += dpp_from<DPP_XOR1>(v0);
    v0 += dpp_from<DPP_XOR2>(v0);
    v0 += dpp_from<DPP_HALF_MIRROR>(v0);
    if (want_kkt) {
        v1 = nan_max(v1, dpp_from<DPP_XOR1>(v1));
        v1 = nan_max(v1, dpp_from<DPP_XOR2>(v1));
        v1 = nan_max(v1, dpp_from<DPP_HALF_MIRROR>(v1));
    }
    // (all eight lanes 8 q .. 8 q + 7 hold them: one store writes every copy)
    if (lane < 8 * NPART && (lane & 7) < SUM_COPIES)
        store_coherent(ex + (int64_t)((lane & 7) * NPART + (lane >> 3)) * slot_ld + wg,
                       lane >= 8 * (NPART - 1) ? v1 : v0);
    ex += (int64_t)(wg % SUM_COPIES) * NPART * slot_ld;
    // the window's maximum without the entry this step replaces
    const int at = st.fs_last + 1 >= sp.m ? 0 : st.fs_last + 1;
    const LaneWindow win{window, wave_max_all(lane == at ? -__builtin_huge_val() : window),
                         lane, 0.0};
    // every workgroup's sums, in slot order per lane; all values of a lane's slots are
    // re-read together until the last one is there
    double v[NPART] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int j0 = lane; j0 < nwg; j0 += 4 * WAVE) {
        double w[4][NPART];
        bool all;
        int n = 0;
        do {
            all = true;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int j = j0 + b * WAVE;
#pragma unroll
                for (int q = 0; q < NPART; q++)
                    w[b][q] = j < nwg ? load_coherent(ex + (int64_t)q * slot_ld + j) : 0.0;
            }
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int q = 0; q < NPART; q++) all = all && published(w[b][q]);
        } while (!all && ++n < LOOP_SPIN_LIMIT);
        if (!all) {
            flags[1] = 1;
            w[0][0] = __builtin_nan("");
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
#pragma unroll
            for (int q = 0; q < NPART - 1; q++) v[q] += w[b][q];
            v[NPART - 1] = nan_max(v[NPART - 1], w[b][NPART - 1]);
        }
    }
    const double tot = wave_sum4(v[0], v[1], v[2], v[3]);
    v[0] = lane_value(tot, ROW_A);
    v[1] = edge_scale * lane_value(tot, ROW_B);
    v[2] = -lane_value(tot, ROW_C) / a_dir;
    v[3] = 0.5 * lane_value(tot, ROW_D);
    v[4] = want_kkt ? wave_max_all(v[4]) : -1.0;  // -1: not evaluated on this pass
    step_core(sample_eps, st, win, v, sp);
    if (lane == 0) {
        sh.a_apply = st.alpha_apply;
        sh.b_apply = st.beta_apply;
        sh.a_dir = st.alpha_dir;
        sh.it = st.it;
        sh.active = st.active;
    }
}

// max |gamma - P(gamma - s g)| over a thread's owned steps (the natural KKT residual)
template <typename S, typename C, int K, int CH, typename Exch>
__device__ __forceinline__ C chunk_kkt(const TileCtx<S, C, K> &cx, int64_t t0, bool owner,
                                       const C (&Q)[K][CH], const C (&G)[K][CH], Exch exch) {
    C gl[K], gr[K], g[K][CH], r = C(0);
    exch(G, gl, gr);
#pragma unroll
    for (int k = 0; k < K; k++) lap_half<C, CH>(G[k], gl[k], gr[k], t0, cx.T, false, g[k]);
#pragma unroll
    for (int c = 0; c < CH; c++) {
        C z[K];
#pragma unroll
        for (int k = 0; k < K; k++)
            z[k] = G[k][c] - cx.s_kkt * (C(2) * cx.alpha * g[k][c] + Q[k][c]);
        project_simplex<K, C>(z);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const C d = fabs(G[k][c] - z[k]);
            if (t0 + c < cx.T) r = (d > r || d != d) ? d : r;
        }
    }
    return owner ? r : C(0);
}

template <typename S, typename C, int K, int CH, int NW>
__global__ __launch_bounds__(NW *WAVE) void spg_loop_1d(LoopArgs A) {
    using L = LoopShape<S, K, CH>;
    constexpr int HT = L::HT, TILE = L::TILE, KS = L::KS, HE = L::HE, ROW = L::ROW, EDGE = L::EDGE;
    using VT = V16<S>;
    constexpr int VW = VT::n;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ LoopShared sh;

    const int nwg = gridDim.x, wg = blockIdx.x;
    const int lane = threadIdx.x & (WAVE - 1), wave = uni((int32_t)(threadIdx.x / WAVE));
    const int tile0 = wg * A.tpw;
    const int ntl = A.ntiles - tile0 < A.tpw ? A.ntiles - tile0 : A.tpw;  // this workgroup's tiles

    S *rows = reinterpret_cast<S *>(lds);                             // [ntl][KS + 1][ROW]
    S *edges = rows + (size_t)A.tpw * (KS + 1) * ROW;                 // [2][tpw + 2][2][EDGE]
    uint8_t *obs_bits = reinterpret_cast<uint8_t *>(edges + (size_t)2 * (A.tpw + 2) * 2 * EDGE);
    // edge `side` (0: first owned steps, 1: last) of local tile lt; -1 and ntl: the neighbouring
    // workgroups' tiles
    auto edge = [&](int par, int lt, int side) {
        return edges + ((size_t)(par * (A.tpw + 2) + lt + 1) * 2 + side) * EDGE;
    };

    TileCtx<S, C, K> cx;
    make_tile_ctx<S, C, K>(A.p, A.p.desc[0], A.p.state[0], cx);
    if (A.kkt_last) cx.want_kkt = false;
    const double sample_eps = uni(A.p.desc[0].alpha) * uni(A.p.desc[0].s_kkt);
    const int kkt_every = A.p.kkt_every > 0 ? A.p.kkt_every : 1;

    LoopState st{};
    double window = 0.0;
    if (wave == 0) loop_load_state(A.p.state[0], A.p.sp.m, lane, st, window);
    const int slot_ld = slot_stride(nwg);
    if (threadIdx.x < 8 * NPART) sh.red[threadIdx.x >> 3][threadIdx.x & 7] = 0.0;
    if (threadIdx.x == 0) sh.parity = A.p.state[0].parity ^ 1;
    // the series ends where no neighbouring workgroup is: zero halos there
    for (int i = threadIdx.x; i < 2 * 2 * EDGE; i += NW * WAVE) {
        const int par = i / (2 * EDGE), r = i - par * 2 * EDGE;
        edge(par, -1, 0)[r] = S(0);
        edge(par, ntl, 0)[r] = S(0);
    }
    __syncthreads();

    const bool owner = lane >= HT && lane < WAVE - HT;
    auto exch = [](const C(&v)[K][CH], C(&l)[K], C(&r)[K]) {
        exchange_edges<C, K, CH, WAVE>(v, nullptr, l, r);
    };

    // gamma rows of a local tile: owned steps from its rows, halo steps from the neighbours' edges
    auto load_tile = [&](int lt, int par, C(&G)[K][CH]) {
        const S *g = owner ? rows + (size_t)lt * (KS + 1) * ROW + lane * CH
                           : (lane < HT ? edge(par, lt - 1, 1) + lane * CH
                                        : edge(par, lt + 1, 0) + (lane - (WAVE - HT)) * CH);
        const int stride = owner ? ROW : HE;
#pragma unroll
        for (int k = 0; k < KS; k++) {
#pragma unroll
            for (int q = 0; q < CH / VW; q++) {
                const typename VT::type v =
                    *reinterpret_cast<const typename VT::type *>(g + k * stride + q * VW);
#pragma unroll
                for (int i = 0; i < VW; i++) G[k][q * VW + i] = C(VT::get(v, i));
            }
        }
    };
    // data term of a local tile, from its data row in LDS or the explicit b in device memory
    auto load_data_term = [&](int lt, int64_t t0, C(&Q)[K][CH]) {
        if (cx.br) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                load_chunk<S, C, CH>(cx.br + k * cx.ld, t0, cx.T, cx.ld, Q[k]);
#pragma unroll
                for (int c = 0; c < CH; c++) Q[k][c] = -Q[k][c];
            }
        } else {
            const S *xrow = rows + ((size_t)lt * (KS + 1) + KS) * ROW + lane * CH;
            C X[CH];
#pragma unroll
            for (int q = 0; q < CH / VW; q++) {
                const typename VT::type v =
                    *reinterpret_cast<const typename VT::type *>(xrow + q * VW);
#pragma unroll
                for (int i = 0; i < VW; i++) X[q * VW + i] = C(VT::get(v, i));
            }
            const unsigned bits = obs_bits[lt * WAVE + lane];
            bool obs[CH];
#pragma unroll
            for (int c = 0; c < CH; c++) obs[c] = (bits >> c) & 1u;
            chunk_data_term<C, K, CH>(cx.theta, cx.bscale, X, obs, Q);
        }
    };

    int e = 0;
    for (; e < A.epochs; e++) {
        double acc[NPART] = {0.0, 0.0, 0.0, 0.0, 0.0};
        const int par = e & 1;
        double *ex = A.ex + L::epoch_words(nwg) * e;  // [sum][workgroup], then the edges
        double *ex_edges = ex + sum_words(nwg);
        for (int lt = wave; lt < ntl; lt += NW) {
            const int tile = tile0 + lt;
            const int64_t t0 = (int64_t)tile * TILE - (int64_t)HT * CH + (int64_t)lane * CH;
            S *trow = rows + (size_t)lt * (KS + 1) * ROW + lane * CH;
            auto levels = [&](auto interior_tile) {
                constexpr bool INT = decltype(interior_tile)::value;
                C G[K][CH], Q[K][CH], G1[K][CH];
                if (e == 0) {
                    // the first iteration of a launch reads device memory
#pragma unroll
                    for (int k = 0; k < KS; k++)
                        load_chunk<S, C, CH, INT>(cx.src + k * cx.ld, t0, cx.T, cx.ld, G[k]);
                    C X[CH];
                    load_chunk<S, C, CH, INT>(cx.xr, t0, cx.T, cx.ld, X);
                    unsigned bits = 0;
#pragma unroll
                    for (int c = 0; c < CH; c++) {
                        const int64_t t = t0 + c;
                        bool o = INT || (t >= 0 && t < cx.T);
                        if (o && cx.heldout) o = cx.heldout[t] == 0;
                        bits |= o ? 1u << c : 0u;
                        trow[KS * ROW + c] = S(X[c]);
                    }
                    obs_bits[lt * WAVE + lane] = (uint8_t)bits;
                } else {
                    load_tile(lt, par, G);
                }
                if (KS < K) {
                    if (cx.first)
                        load_chunk<S, C, CH, INT>(cx.src + (K - 1) * cx.ld, t0, cx.T, cx.ld,
                                                  G[K - 1]);
                    else
                        rebuild_last_row<C, K, CH, INT>(t0, cx.T, G);
                }
                load_data_term(lt, t0, Q);
                LevelSums<C> p;
                pass_levels<S, C, K, CH, INT>(cx, t0, owner, Q, G, exch, []() {}, G1, p);
                if (owner) {
                    // gamma_i to the tile's rows (0 past the end, as the halo loads give it)
#pragma unroll
                    for (int k = 0; k < KS; k++) {
#pragma unroll
                        for (int c = 0; c < CH; c++)
                            if (!INT && t0 + c >= cx.T) G1[k][c] = C(0);
#pragma unroll
                        for (int q = 0; q < CH / VW; q++) {
                            typename VT::type v;
#pragma unroll
                            for (int i = 0; i < VW; i++) VT::set(v, i, S(G1[k][q * VW + i]));
                            *reinterpret_cast<typename VT::type *>(trow + k * ROW + q * VW) = v;
                        }
                    }
                    // and its outer steps to the neighbours: LDS, and the exchange area at the
                    // ends of the workgroup
                    auto put = [&](int side, int at) {
                        S *o = edge(par ^ 1, lt, side) + at;
                        const bool out = side == 0 ? (lt == 0 && wg > 0)
                                                   : (lt == ntl - 1 && wg < nwg - 1);
                        double *og = ex_edges + ((int64_t)wg * 2 + side) * EDGE + at;
#pragma unroll
                        for (int k = 0; k < KS; k++) {
#pragma unroll
                            for (int c = 0; c < CH; c++) {
                                o[k * HE + c] = S(G1[k][c]);
                                if (out) store_coherent(og + k * HE + c, (double)S(G1[k][c]));
                            }
                        }
                    };
                    if (lane < 2 * HT) put(0, (lane - HT) * CH);
                    if (lane >= WAVE - 2 * HT) put(1, (lane - (WAVE - 2 * HT)) * CH);
                }
                acc[0] += (double)p.dd;
                acc[1] += (double)p.dad;
                acc[2] += (double)p.dd + (double)p.off;
                acc[3] += (double)p.f;
                const double kk = (double)p.kkt;
                acc[4] = nan_max(acc[4], kk);
            };
            if (tile_is_interior<S, C, K, CH, WAVE>(tile, cx.T))
                levels(std::true_type{});
            else
                levels(std::false_type{});
        }
        loop_sums<NW>(sh, acc, cx.want_kkt, lane, wave);
        lds_barrier();
        if (wave == 0)
            loop_step(sh, cx.want_kkt, 2.0 * (double)cx.alpha, (double)cx.a_dir, sample_eps, ex, slot_ld,
                      nwg, wg, lane, st, window, A.p.sp, A.flags);
        if (wave == NW - 1) {
            // the neighbouring workgroups' edges of this iteration
            for (int i = lane; i < 2 * EDGE; i += WAVE) {
                const int side = i / EDGE, r = i - side * EDGE;  // 0: from the left, 1: the right
                const int nb = side == 0 ? wg - 1 : wg + 1;
                if (nb < 0 || nb >= nwg) continue;
                const double *src = ex_edges + ((int64_t)nb * 2 + (side ^ 1)) * EDGE + r;
                edge(par ^ 1, side == 0 ? -1 : ntl, side ^ 1)[r] =
                    S(await_value(src, A.flags + 1));
            }
        }
        lds_barrier();
        cx.a_apply = uni(C(sh.a_apply));
        cx.b_apply = uni(C(sh.b_apply));
        cx.a_dir = uni(C(sh.a_dir));
        cx.first = false;
        cx.need_f = A.p.need_f;
        cx.want_kkt = !A.kkt_last && uni(sh.it) % kkt_every == 0;
        if (uni(sh.active) == 0) break;
    }
    // the residual of the iterate that stopped, where no iteration asked for it
    if (A.kkt_last && uni(sh.active) == 0) {
        double kkt = 0.0;
        for (int lt = wave; lt < ntl; lt += NW) {
            const int64_t t0 = (int64_t)(tile0 + lt) * TILE - (int64_t)HT * CH + (int64_t)lane * CH;
            C G[K][CH], Q[K][CH], p;
            load_tile(lt, (e + 1) & 1, G);
            if (KS < K) rebuild_last_row<C, K, CH, false>(t0, cx.T, G);
            load_data_term(lt, t0, Q);
            p = chunk_kkt<S, C, K, CH>(cx, t0, owner, Q, G, exch);
            kkt = nan_max(kkt, (double)p);
        }
        kkt = wave_max_all(kkt);
        if (lane == 0) sh.red[4][wave] = kkt;
        __syncthreads();
        double *ex = A.ex + L::epoch_words(nwg) * (e + 1);
        if (wave == 0) {
            kkt = 0.0;
#pragma unroll
            for (int w = 0; w < NW; w++) kkt = nan_max(kkt, sh.red[4][w]);
            if (lane == 0) store_coherent(ex + wg, kkt);
            if (wg == 0) {
                for (int j = lane; j < nwg; j += WAVE)
                    kkt = nan_max(kkt, await_value(ex + j, A.flags + 1));
                st.kkt = wave_max_all(kkt);
            }
        }
    }
    // the iterate to the launch's other buffer: K rows, the last rebuilt as complete_last_row
    S *dst = reinterpret_cast<S *>(uni(sh.parity) ? A.p.gamma1 : A.p.gamma0) + uni(A.p.desc[0].goff);
    for (int lt = wave; lt < ntl; lt += NW) {
        const int64_t t0 = (int64_t)(tile0 + lt) * TILE - (int64_t)HT * CH + (int64_t)lane * CH;
        const S *trow = rows + (size_t)lt * (KS + 1) * ROW + lane * CH;
        if (!owner) continue;
        S v[K][CH];
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int c = 0; c < CH; c++) v[k][c] = trow[k * ROW + c];
        if (KS < K) {
#pragma unroll
            for (int c = 0; c < CH; c++) {
                S r = S(1);
#pragma unroll
                for (int k = 0; k < K - 1; k++) r -= v[k][c];
                v[K - 1][c] = r > S(0) ? r : S(0);
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
#pragma unroll
            for (int q = 0; q < CH / VW; q++) {
                const int64_t t = t0 + q * VW;
                if (t + VW <= cx.T) {
                    typename VT::type o;
#pragma unroll
                    for (int i = 0; i < VW; i++) VT::set(o, i, v[k][q * VW + i]);
                    *reinterpret_cast<typename VT::type *>(dst + k * cx.ld + t) = o;
                } else {
#pragma unroll
                    for (int i = 0; i < VW; i++)
                        if (t + i < cx.T) dst[k * cx.ld + t + i] = v[k][q * VW + i];
                }
            }
        }
    }
    if (wg == 0 && wave == 0) {
        st.parity = uni(sh.parity);
        loop_put_state(A.p.state[0], A.p.sp.m, lane, st, window);
        loop_put_state(*A.out, A.p.sp.m, lane, st, window);
        if (lane == 0) {
            A.flags[0] = st.active;
        }
    }
}

}  // namespace pasc
