// Persistent SPG loop for one image that fits on chip (the image pass's problem, img_kernels.h, in
// the manner of loop_kernels.h): one launch runs many iterations with the iterate in registers.
//
// The image pass walks its rows one after the other, with a launch, the first rows' loads and the
// hand-over around the walk.  Here a workgroup of NW waves owns a tile of 64 columns x NW*RPW
// rows; lane = column, each wave holds RPW rows of gamma_i and p_i in registers (their last
// components in LDS), and q too or prefetches it a row ahead.  Left and right neighbours come from
// the adjacent lanes, rows above and below from registers or, between waves, LDS; no node is
// computed twice.  us per iteration, image pass / here (FP64): 250 x 150, K = 2 13.4 / 5.3;
// 512 x 512, K = 3 16.4 / 7.9; 1024 x 1024, K = 2 / 3 / 4 19.7 / 23.7 / 29.5 against 9.7 / 12.1 /
// 15.5 (FP32, K = 4: 25 / 12.4); 300 x 200, K = 8 36 / 8.8.  Issue bounds the large ones (270 - 370
// instructions a row, two waves per SIMD), the two exchanges (~2 us each) the small ones.
// What the layout costs when left out: a row's q loaded where it is used 16 us of 26 at 1024 x 1024,
// K = 4; reads of the columns beyond the tile under a lane condition, eight branches a row;
// the outer columns published lane by lane, 128 partial stores a wave.
// Between workgroups an iteration exchanges the tiles' outer rows and columns of p_i: the owner of a
// halo node (one thread each) keeps its gamma and advances it as its owner does.  So an
// iteration is
//   1. gamma_i = gamma_{i-1} + beta (p_{i-1} - gamma_{i-1}) on the tile and its halo;
//   2. g_i, p_i and the node sums of the tile; the tile's outer p_i to the neighbours;
//   3. the neighbours' p_i, then the edge sums (d_a - d_b)^2, each edge with its upper or left end;
//   4. the sums and the step (loop_sums, loop_step).
// The exchanged rows lie in four sets used in turn.  While a workgroup publishes into one, it marks
// its places of the set after the next empty: that set's last readers ended before they published
// the sums of two iterations before, which this workgroup has read.  The marks are complete
// (vmcnt) before it publishes anything of the next iteration, and a reader turns to that set
// only with that iteration's sums.
// Every node's arithmetic is the image pass's; the sums differ in order only.
#pragma once

#include "img_kernels.h"
#include "loop_kernels.h"

namespace pasc {

constexpr int IMG_SETS = 4;

struct ImgLoopArgs {
    ImgArgs p;           // buffers, descriptor, state, sizes (grp, part, counters not used)
    double *ex;          // (epochs + 1) x sums of nwg workgroups, then IMG_SETS sets of edges
    double *edges;
    InstState *out;      // pinned host copy of the final state
    int32_t *flags;      // pinned: [0] still active, [1] a wait ran out
    int32_t nct;         // tiles across the image
    int32_t epochs;
    int32_t kkt_last;    // as LoopArgs
    int32_t need_f;
};

// q in registers too (96 of the 256 a thread of 8 waves has), else read again by every iteration
template <typename S>
constexpr bool img_loop_q(int K, int rpw) {
    return 3 * K * (int)(sizeof(S) / 4) * rpw <= 96;
}

// Rows a wave holds at most (gamma and p, 2 K values a row, besides what the projection of a row
// needs): more spill.
template <typename S>
constexpr int img_loop_rows(int K) {
    return sizeof(S) == 8 ? (K <= 4 ? 8 : K == 5 ? 4 : K == 6 ? 2 : 1) : (K <= 5 ? 8 : 4);
}

template <typename S, int K, int NW, int RPW>
struct ImgLoopShape {
    static constexpr int TH = NW * RPW;
    static constexpr int EDGE = K * (2 * WAVE + 2 * TH);  // values a workgroup publishes
    // LDS: gamma of every wave's first and last row, d of its first; gamma, p and d of the halo
    static constexpr int HN = 2 * WAVE + 2 * TH;  // halo nodes: above, below, left, right
    // and the tile's last rows of gamma and p; p of its outer columns
    static constexpr size_t LDS =
        sizeof(S) * ((size_t)K * (NW * 3 * WAVE + 3 * HN) + 2 * TH * WAVE + 2 * K * TH);
};

template <typename S, int K, int NW, int RPW>
__global__ __launch_bounds__(NW *WAVE) void img_loop(ImgLoopArgs A) {
    using C = S;
    using L = ImgLoopShape<S, K, NW, RPW>;
    constexpr int KS = stored_rows<K>(), TH = L::TH, HN = L::HN;
    constexpr bool QREG = img_loop_q<S>(K, RPW);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ LoopShared sh;
    C *erow = reinterpret_cast<C *>(lds);          // [NW][2][K][64] gamma of the first and last row
    C *drow = erow + NW * 2 * K * WAVE;            // [NW][K][64] d of the first row
    C *hgam = drow + NW * K * WAVE, *hp = hgam + K * L::HN, *hd = hp + K * L::HN;  // [K][HN]
    C *lrow = hd + K * L::HN + (threadIdx.x / WAVE) * RPW * WAVE + (threadIdx.x & (WAVE - 1));
    C *prow = lrow + TH * WAVE;
    C *pcol = hd + K * L::HN + 2 * TH * WAVE + (threadIdx.x / WAVE) * 2 * K * RPW;  // [2][K][RPW]

    const int nwg = gridDim.x, wg = blockIdx.x, nct = A.nct, nrt = nwg / nct;
    const int ct = wg % nct, rt = wg / nct;
    const int lane = threadIdx.x & (WAVE - 1), wave = uni((int32_t)(threadIdx.x / WAVE));
    const int W = A.p.width, H = A.p.height;
    const int col = ct * WAVE + lane, r0 = rt * TH, y0 = r0 + wave * RPW;
    const bool colin = col < W;
    const int slot_ld = slot_stride(nwg);

    ImgCtx<S, C, K> cx;
    make_img_ctx<S, C, K>(A.p, A.p.desc[0], A.p.state[0], cx);
    if (A.kkt_last) cx.want_kkt = false;
    const uint32_t ld = cx.ld;
    const double sample_eps = uni(A.p.desc[0].alpha) * uni(A.p.desc[0].s_kkt);
    const int kkt_every = A.p.kkt_every > 0 ? A.p.kkt_every : 1;
    bool first = uni(A.p.state[0].first) != 0;
    bool need_f = A.need_f || first;
    LoopState st{};
    double window = 0.0;
    if (wave == 0) loop_load_state(A.p.state[0], A.p.sp.m, lane, st, window);
    if (threadIdx.x < 8 * NPART) sh.red[threadIdx.x >> 3][threadIdx.x & 7] = 0.0;
    if (threadIdx.x == 0) sh.parity = A.p.state[0].parity ^ 1;

    // the halo node of this thread: side 0 above, 1 below, 2 left, 3 right; place `at` on the side
    const int u = threadIdx.x;
    const int side = u < WAVE ? 0 : u < 2 * WAVE ? 1 : u < 2 * WAVE + TH ? 2 : 3;
    const int at = side == 0 ? u : side == 1 ? u - WAVE : side == 2 ? u - 2 * WAVE : u - 2 * WAVE - TH;
    const int hx = side < 2 ? ct * WAVE + at : side == 2 ? ct * WAVE - 1 : ct * WAVE + WAVE;
    const int hy = side == 0 ? r0 - 1 : side == 1 ? r0 + TH : r0 + at;
    const bool halo = u < 2 * WAVE + 2 * TH && hx >= 0 && hx < W && hy >= 0 && hy < H;
    const int nb = side == 0 ? wg - nct : side == 1 ? wg + nct : side == 2 ? wg - 1 : wg + 1;
    // where the neighbour publishes it: its opposite side, at the same place
    // (a column is published wave by wave, [K][RPW] each)
    const int in_col = K * (at - at % RPW) + at % RPW;
    const int src_off = side == 0 ? K * WAVE + at : side == 1 ? at
                        : side == 2 ? K * (2 * WAVE + TH) + in_col : K * 2 * WAVE + in_col;
    const int src_ld = side < 2 ? WAVE : RPW;

    // gamma (K - 1 rows, the last in LDS), p and q of this lane's column in the wave's rows
    C gam[RPW][KS], p[RPW][KS], q[QREG ? RPW : 1][K];
#pragma unroll
    for (int j = 0; j < RPW; j++) {
        const int y = y0 + j;
        const bool in = colin && y < H;
        const uint32_t n = in ? (uint32_t)(y * W + col) : 0u;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            gam[j][k] = in ? at32(cx.src, k * ld + n) : C(0);
            p[j][k] = in && !first ? at32(cx.pprev, k * ld + n) : C(0);
        }
        if (first) {  // gamma_0 is projected
            C v[K];
#pragma unroll
            for (int k = 0; k < K; k++) v[k] = in ? at32(cx.src, k * ld + n) : C(0);
            project_simplex<K, C>(v);
#pragma unroll
            for (int k = 0; k < KS; k++) gam[j][k] = v[k];
            if (KS < K) lrow[j * WAVE] = v[K - 1];
        }
        if (QREG)
#pragma unroll
            for (int k = 0; k < K; k++) q[QREG ? j : 0][k] = in ? at32(cx.q, k * ld + n) : C(0);
    }
    {
        const uint32_t n = halo ? (uint32_t)(hy * W + hx) : 0u;
        if (halo) {
            C v[K];
#pragma unroll
            for (int k = 0; k < K; k++) {
                v[k] = k < KS || first ? at32(cx.src, k * ld + n) : C(0);
                hp[k * HN + u] = k < KS && !first ? at32(cx.pprev, k * ld + n) : C(0);
            }
            if (first) project_simplex<K, C>(v);
#pragma unroll
            for (int k = 0; k < K; k++) hgam[k * HN + u] = v[k];
        } else if (u < HN) {
#pragma unroll
            for (int k = 0; k < K; k++) hgam[k * HN + u] = C(0);  // finite: it meets weight 0
        }
    }
    // gamma_i of a node from gamma_{i-1} and p_{i-1} (img_gamma's arithmetic)
    auto advance = [&](C(&g)[KS], C &l, const C *pp) {
        C v[K];
        if (cx.beta == C(1)) {
#pragma unroll
            for (int k = 0; k < KS; k++) v[k] = pp[k];
        } else {
#pragma unroll
            for (int k = 0; k < KS; k++) v[k] = g[k] + cx.beta * (pp[k] - g[k]);
        }
        if (KS < K) v[K - 1] = last_row(v);
#pragma unroll
        for (int k = 0; k < KS; k++) g[k] = v[k];
        if (KS < K) l = v[K - 1];
    };
    // p_i of row j
    auto node_p = [&](int j, C(&v)[K]) {
#pragma unroll
        for (int k = 0; k < KS; k++) v[k] = p[j][k];
        if (KS < K) v[K - 1] = prow[j * WAVE];
    };
    // gamma_i of row j
    auto node = [&](int j, C(&v)[K]) {
#pragma unroll
        for (int k = 0; k < KS; k++) v[k] = gam[j][k];
        if (KS < K) v[K - 1] = lrow[j * WAVE];
    };
    const int side_at = 2 * WAVE + wave * RPW + (lane == 0 ? 0 : TH);
    const C wl = col > 0 ? C(1) : C(0), wr = col < W - 1 ? C(1) : C(0);
    // the Laplacian at row j of this lane's column, in the walk order up, left, right, down
    auto laplacian = [&](int j, int y, const C(&gc)[K], C(&lap)[K]) {
        const C wu = y > 0 ? C(1) : C(0), wd = y + 1 < H ? C(1) : C(0);
        C up[K], dn[K];
        if (j > 0) node(j > 0 ? j - 1 : 0, up);
        if (j < RPW - 1) node(j < RPW - 1 ? j + 1 : 0, dn);
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (j == 0)
                up[k] = wave > 0 ? erow[((wave - 1) * 2 + 1) * K * WAVE + k * WAVE + lane]
                                 : hgam[k * HN + lane];
            if (j == RPW - 1)
                dn[k] = wave < NW - 1 ? erow[(wave + 1) * 2 * K * WAVE + k * WAVE + lane]
                                      : hgam[k * HN + WAVE + lane];
            // beyond the tile's columns: one read serves lane 0 (left halo) and lane 63 (right)
            const C beyond = hgam[k * HN + side_at + j];
            C gl = dpp_shift<DPP_WAVE_SHR1>(gc[k]), gr = dpp_shift<DPP_WAVE_SHL1>(gc[k]);
            gl = lane == 0 ? beyond : gl;
            gr = lane == WAVE - 1 ? beyond : gr;
            C l = wu * (gc[k] - up[k]);
            l = l + wl * (gc[k] - gl);
            l = l + wr * (gc[k] - gr);
            l = l + wd * (gc[k] - dn[k]);
            lap[k] = l;
        }
    };
    // q of a row, from registers or from the caches (columns past the image read the last one's)
    const int qcol = colin ? col : W - 1;
    C qn[K];  // of the next row
    auto fetch_q = [&](int y) {
        const uint32_t n = (uint32_t)((y < H ? y : H - 1) * W + qcol);
#pragma unroll
        for (int k = 0; k < K; k++) qn[k] = at32(cx.q, k * ld + n);
    };
    auto row_q = [&](int j, int y, C(&v)[K]) {
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = QREG ? q[QREG ? j : 0][k] : qn[k];
        if (!QREG && j + 1 < RPW) fetch_q(y + 1);
    };
    if (!QREG) fetch_q(y0);
    __syncthreads();

    bool fresh = first;  // gamma_0 stands
    int e = 0;
    for (; e < A.epochs; e++) {
        double *ex = A.ex + sum_words(nwg) * e;
        double *set = A.edges + (int64_t)(e % IMG_SETS) * nwg * L::EDGE;
        double *next = A.edges + (int64_t)((e + 2) % IMG_SETS) * nwg * L::EDGE;
        double *mine = set + (int64_t)wg * L::EDGE, *empty = next + (int64_t)wg * L::EDGE;
        double acc[NPART] = {0.0, 0.0, 0.0, 0.0, 0.0};
        // recomputed in every iteration: kept, the rows' conditions would spill
        int yb = y0;
        asm volatile("" : "+s"(yb));
        // 1. gamma_i
#pragma unroll
        for (int j = 0; j < RPW; j++) {
            if (!fresh) {
                C l = C(0);
                advance(gam[j], l, p[j]);
                if (KS < K) lrow[j * WAVE] = l;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (halo && !fresh) {
            C g[KS], l = hgam[(K - 1) * HN + u], pp[KS];
#pragma unroll
            for (int k = 0; k < KS; k++) {
                g[k] = hgam[k * HN + u];
                pp[k] = hp[k * HN + u];
            }
            advance(g, l, pp);
#pragma unroll
            for (int k = 0; k < K; k++) hgam[k * HN + u] = k < KS ? g[k < KS ? k : 0] : l;
        }
        {
            C top[K], bot[K];
            node(0, top);
            node(RPW - 1, bot);
#pragma unroll
            for (int k = 0; k < K; k++) {
                erow[wave * 2 * K * WAVE + k * WAVE + lane] = top[k];
                erow[(wave * 2 + 1) * K * WAVE + k * WAVE + lane] = bot[k];
            }
        }
        lds_barrier();
        // 2. the direction and the node sums
#pragma unroll
        for (int j = 0; j < RPW; j++) {
            const int y = yb + j;
            if (y >= H) break;
            C gc[K], lap[K], g[K], qv[K], yv[K], z[K], pv[K];
            row_q(j, y, qv);
            node(j, gc);
            laplacian(j, y, gc, lap);
#pragma unroll
            for (int k = 0; k < K; k++) {
                g[k] = cx.alpha * lap[k] + qv[k];
                yv[k] = gc[k] - cx.a_dir * g[k];
                pv[k] = yv[k];
                z[k] = gc[k] - cx.s_kkt * g[k];
            }
            __builtin_amdgcn_sched_barrier(0);
            const C tau = project_simplex<K, C>(pv);
#pragma unroll
            for (int k = 0; k < KS; k++) p[j][k] = pv[k];
            if (KS < K) prow[j * WAVE] = pv[K - 1];
            if (lane == 0 || lane == WAVE - 1) {
#pragma unroll
                for (int k = 0; k < K; k++) pcol[(lane == 0 ? 0 : K * RPW) + k * RPW + j] = pv[k];
            }
            __builtin_amdgcn_sched_barrier(0);
            double dd = 0.0, off = 0.0, fq = 0.0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                const C d = pv[k] - gc[k];
                if (j == 0) drow[wave * K * WAVE + k * WAVE + lane] = d;
                dd += (double)d * (double)d;
                // the off-support term of <g, d>: (tau - y_k) gamma_k where y_k <= tau
                const C o = tau - yv[k];
                off += (double)(o > C(0) ? o : C(0)) * (double)gc[k];
                fq += ((double)g[k] + (double)qv[k]) * (double)gc[k];
            }
            acc[0] += colin ? dd : 0.0;
            acc[2] += colin ? dd + off : 0.0;
            acc[3] += colin ? fq : 0.0;
            if (cx.want_kkt) {
                project_simplex<K, C>(z);
                double m = 0.0;
#pragma unroll
                for (int k = 0; k < K; k++) m = nan_max(m, fabs((double)gc[k] - (double)z[k]));
                acc[4] = nan_max(acc[4], colin ? m : 0.0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // the tile's outer p_i to the neighbours, this workgroup's places of the set after the next
        // empty (last iteration's marks are complete)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const double none = __builtin_bit_cast(double, PART_EMPTY);
        auto publish = [&](int off, int stride, const C(&v)[K]) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                store_coherent(mine + off + k * stride, (double)v[k]);
                store_coherent(empty + off + k * stride, none);
            }
        };
        if (wave == 0 && rt > 0 && colin) {
            C v[K];
            node_p(0, v);
            publish(lane, WAVE, v);
        }
        if (wave == NW - 1 && rt < nrt - 1 && colin) {
            C v[K];
            node_p(RPW - 1, v);
            publish(K * WAVE + lane, WAVE, v);
        }
        for (int i = lane; i < 2 * K * RPW; i += WAVE) {  // (this wave's own writes: no barrier)
            const int right = i >= K * RPW, o = i - right * K * RPW;
            if ((right ? ct < nct - 1 : ct > 0) && yb + o % RPW < H) {
                const int off = K * (2 * WAVE + right * TH + wave * RPW) + o;
                store_coherent(mine + off, (double)pcol[i]);
                store_coherent(empty + off, none);
            }
        }
        // 3. the neighbours' p_i
        if (halo) {
            const double *src = set + (int64_t)nb * L::EDGE + src_off;
            double v[K];
            bool all;
            int n = 0;
            do {
                all = true;
#pragma unroll
                for (int k = 0; k < K; k++) v[k] = load_coherent(src + k * src_ld);
#pragma unroll
                for (int k = 0; k < K; k++) all = all && published(v[k]);
            } while (!all && ++n < LOOP_SPIN_LIMIT);
            if (!all) A.flags[1] = 1;
#pragma unroll
            for (int k = 0; k < K; k++) {
                hp[k * HN + u] = C(v[k]);
                hd[k * HN + u] = C(v[k]) - hgam[k * HN + u];
            }
        }
        lds_barrier();
        {
            C d[K], dn[K], gc[K], pv[K];
            node(0, gc);
            node_p(0, pv);
#pragma unroll
            for (int k = 0; k < K; k++) d[k] = pv[k] - gc[k];
#pragma unroll
            for (int j = 0; j < RPW; j++) {
                const int y = yb + j;
                if (y >= H) break;
                double eh = 0.0, ev = 0.0;
                if (j < RPW - 1) {
                    node(j < RPW - 1 ? j + 1 : 0, gc);
                    node_p(j < RPW - 1 ? j + 1 : 0, pv);
                }
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const C beyond = hd[k * HN + 2 * WAVE + TH + wave * RPW + j];
                    C dr = dpp_shift<DPP_WAVE_SHL1>(d[k]);
                    dr = lane == WAVE - 1 ? beyond : dr;
                    if (j < RPW - 1)
                        dn[k] = pv[k] - gc[k];
                    else
                        dn[k] = wave < NW - 1 ? drow[(wave + 1) * K * WAVE + k * WAVE + lane]
                                              : hd[k * HN + WAVE + lane];
                    const double e1 = (double)d[k] - (double)dr;
                    const double e2 = (double)d[k] - (double)dn[k];
                    eh += e1 * e1;
                    ev += e2 * e2;
                }
                acc[1] += col < W - 1 ? eh : 0.0;
                acc[1] += colin && y + 1 < H ? ev : 0.0;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < K; k++) d[k] = dn[k];
            }
        }
        // 4. the sums and the step
        if (!need_f) acc[3] = 0.0;
        // an overflow (of FP32: its f comes from the step, which would carry an infinity on) ends the
        // solve as a NaN does; the image pass meets it as 0 * inf in its halo columns
        acc[2] += 0.0 * acc[2];
        acc[3] += 0.0 * acc[3];
        loop_sums<NW>(sh, acc, cx.want_kkt, lane, wave);
        if (!QREG) fetch_q(y0);  // of the next iteration
        lds_barrier();
        if (wave == 0)
            loop_step(sh, cx.want_kkt, cx.alpha_d, cx.a_dir_d, sample_eps, ex, slot_ld, nwg, wg, lane, st,
                      window, A.p.sp, A.flags);
        lds_barrier();
        cx.beta = uni(C(sh.b_apply));
        cx.a_dir = uni(C(sh.a_dir));
        cx.a_dir_d = (double)cx.a_dir;
        fresh = false;
        need_f = A.need_f;
        cx.want_kkt = !A.kkt_last && uni(sh.it) % kkt_every == 0;
        if (uni(sh.active) == 0) break;
    }
    // the residual of the iterate that stopped, where no iteration asked for it
    if (A.kkt_last && uni(sh.active) == 0) {
        double kkt = 0.0;
#pragma unroll
        for (int j = 0; j < RPW; j++) {
            const int y = y0 + j;
            if (y >= H) break;
            C gc[K], lap[K], z[K], qv[K];
            row_q(j, y, qv);
            node(j, gc);
            laplacian(j, y, gc, lap);
#pragma unroll
            for (int k = 0; k < K; k++) z[k] = gc[k] - cx.s_kkt * (cx.alpha * lap[k] + qv[k]);
            project_simplex<K, C>(z);
            double m = 0.0;
#pragma unroll
            for (int k = 0; k < K; k++) m = nan_max(m, fabs((double)gc[k] - (double)z[k]));
            kkt = nan_max(kkt, colin ? m : 0.0);
            __builtin_amdgcn_sched_barrier(0);
        }
        kkt = wave_max_all(kkt);
        if (lane == 0) sh.red[4][wave] = kkt;
        __syncthreads();
        double *ex = A.ex + sum_words(nwg) * (e + 1);
        if (wave == 0) {
            kkt = 0.0;
#pragma unroll
            for (int w = 0; w < NW; w++) kkt = nan_max(kkt, sh.red[4][w]);
            if (lane == 0) store_coherent(ex + wg, kkt);
            if (wg == 0) {
                for (int j = lane; j < nwg; j += WAVE) kkt = nan_max(kkt, await_value(ex + j, A.flags + 1));
                st.kkt = wave_max_all(kkt);
            }
        }
    }
    // gamma_i (K rows) and p_i to the launch's other buffers
    const int par = uni(sh.parity);
    const int64_t goff = uni(A.p.desc[0].goff);
    S *dst = reinterpret_cast<S *>(par ? A.p.gamma1 : A.p.gamma0) + goff;
    S *pout = reinterpret_cast<S *>(par ? A.p.dir1 : A.p.dir0) + goff;
#pragma unroll
    for (int j = 0; j < RPW; j++) {
        if (!colin || y0 + j >= H) continue;
        const uint32_t n = (uint32_t)((y0 + j) * W + col);
#pragma unroll
        for (int k = 0; k < KS; k++) {
            at32(dst, k * ld + n) = gam[j][k];
            at32(pout, k * ld + n) = p[j][k];
        }
        if (KS < K) {
            C v[K];
            node(j, v);
            at32(dst, (K - 1) * ld + n) = last_row(v);  // as complete_last_row does
        }
    }
    if (wg == 0 && wave == 0) {
        st.parity = par;
        loop_put_state(A.p.state[0], A.p.sp.m, lane, st, window);
        loop_put_state(*A.out, A.p.sp.m, lane, st, window);
        if (lane == 0) A.flags[0] = st.active;
    }
}

}  // namespace pasc
