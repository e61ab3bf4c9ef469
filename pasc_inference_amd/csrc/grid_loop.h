// Persistent SPG loop for one spatio-temporal grid (T frames of an image, T > 1) that fits on chip:
// the graph kernels' problem (spg_pass_grid_dir / _ad) in the manner of loop_kernels.h.
//
// The graph kernels take three launches per iteration and gather gamma_{i-1} and d_{i-1} of 14
// neighbours per node through branches and 64-bit index arithmetic: 36 us on 60 frames of
// 64 x 48, K = 3, FP64 (here 9.3 in a long launch), 60 on 100 frames of 64 x 64 (12.5).  Here a
// workgroup owns a brick of bx x by x bt nodes; gamma and d of the brick and of the nodes around it
// lie in LDS, q and the node's place in registers, up to NPT nodes a thread.  What is left at 60
// frames, us: node pass 2.2, edges 0.9, gamma 0.6 (LDS reads and FP64 issue), exchange of d 2, sums
// and step 4.  An iteration
//   1. advances gamma on the brick and around it, gamma_i = gamma_{i-1} + beta d_{i-1};
//   2. forms g_i and d_i of the brick and publishes d_i of its outer nodes;
//   3. takes the d_i around it from the bricks that own them (sets and marks as in img_loop.h) and
//      sums the edges, each with its lower node;
//   4. adds up the sums and takes the step (loop_sums, loop_step).
// Every node's arithmetic is the graph kernels'; the sums differ in order only.
#pragma once

#include "img_loop.h"

namespace pasc {

constexpr int GRID_LOOP_NW = 8;                      // waves per workgroup
constexpr int GRID_LOOP_NT = GRID_LOOP_NW * WAVE;
constexpr int GRID_LOOP_HPT = 4;                     // nodes around the brick per thread at most

struct GridLoopArgs {
    GridArgs p;      // buffers, descriptor, data, sizes (state, grp, part not used)
    InstState *state;
    StepParams sp;
    double *ex;      // as ImgLoopArgs
    double *edges;
    InstState *out;
    int32_t *flags;
    int32_t bx, by, bt;  // brick
    int32_t nx, ny;      // bricks across and down
    int32_t epochs;
    int32_t kkt_last;
};

// Nodes of a tile (the brick and the nodes around it) at most.  Also the distance of two components
// in LDS, whatever the brick: a constant that goes into the instructions' offsets.
template <typename S>
constexpr int grid_loop_tile(int K) {
    return (int)((LOOP_LDS_BYTES - 1024) / (sizeof(S) * (K + (K >= 2 ? K - 1 : K))));
}
template <typename S>
constexpr size_t grid_loop_lds(int K) {
    return sizeof(S) * (size_t)(K + (K >= 2 ? K - 1 : K)) * grid_loop_tile<S>(K);
}

template <typename S, int K, int NPT>
__global__ __launch_bounds__(GRID_LOOP_NT) void grid_loop(GridLoopArgs A) {
    using C = S;
    constexpr int KS = stored_rows<K>(), NW = GRID_LOOP_NW, NT = GRID_LOOP_NT, HPT = GRID_LOOP_HPT;
    constexpr int ts = grid_loop_tile<S>(K);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ LoopShared sh;
    const int bx = A.bx, by = A.by, bt = A.bt, nx = A.nx, ny = A.ny;
    const int ex_ = bx + 2, ey_ = by + 2, et_ = bt + 2;       // the brick and the nodes around it
    const int py = ex_, pt = ex_ * ey_;                        // pitches
    C *gam = reinterpret_cast<C *>(lds);                       // [K][ts]
    C *dir = gam + K * ts;                                     // [KS][ts]

    const InstDesc &D = A.p.desc[0];
    const int nwg = gridDim.x, wg = blockIdx.x, tid = threadIdx.x;
    const int lane = tid & (WAVE - 1), wave = uni((int32_t)(tid / WAVE));
    const int W = A.p.geo.width, H = (int)(A.p.geo.R / W), T = (int)A.p.geo.T;
    const int brick = bx * by * bt;
    const int x0 = (wg % nx) * bx, y0 = (wg / nx % ny) * by, t0 = (wg / (nx * ny)) * bt;
    const int slot_ld = slot_stride(nwg);
    const int64_t ld = uni(D.ld), goff = uni(D.goff);
    const C alpha = C(uni(D.alpha)), s_kkt = C(uni(D.s_kkt));
    const double alpha_d = uni(D.alpha), sample_eps = alpha_d * uni(D.s_kkt);
    const bool first = uni(A.state[0].first) != 0;
    const int par0 = uni(A.state[0].parity);
    C beta = C(uni(A.state[0].beta_apply)), a_dir = C(uni(A.state[0].alpha_dir));
    LoopState st{};
    double window = 0.0;
    if (wave == 0) loop_load_state(A.state[0], A.sp.m, lane, st, window);
    if (tid < 8 * NPART) sh.red[tid >> 3][tid & 7] = 0.0;
    if (tid == 0) sh.parity = par0 ^ 1;
    for (int i = tid; i < (K + KS) * ts; i += NT) gam[i] = C(0);  // finite: it meets weight 0
    __syncthreads();

    const S *src = reinterpret_cast<const S *>(par0 ? A.p.gamma1 : A.p.gamma0) + goff;
    const S *dprev = reinterpret_cast<const S *>(par0 ? A.p.dir1 : A.p.dir0) + goff;
    auto load_node = [&](int li, int64_t n) {
        C v[K];
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = k < KS || first ? C(src[k * ld + n]) : C(0);
        if (first) project_simplex<K, C>(v);
#pragma unroll
        for (int k = 0; k < K; k++) gam[k * ts + li] = v[k];
#pragma unroll
        for (int k = 0; k < KS; k++) dir[k * ts + li] = first ? C(0) : C(dprev[k * ld + n]);
    };
    // this thread's nodes: tile index (-1: none), global index, which neighbours exist
    enum { TM = 1, TP = 2, UP = 4, LEFT = 8, RIGHT = 16, DOWN = 32, OUTER = 64 };
    int li[NPT], gn[NPT], has[NPT];
    C q[NPT][K];
    const GridData gd = grid_data(D);
#pragma unroll
    for (int j = 0; j < NPT; j++) {
        const int o = tid + j * NT, ox = o % bx, oy = o / bx % by, ot = o / (bx * by);
        const int x = x0 + ox, y = y0 + oy, t = t0 + ot;
        const bool in = o < brick && x < W && y < H && t < T;
        li[j] = in ? (ot + 1) * pt + (oy + 1) * py + ox + 1 : -1;
        gn[j] = in ? (t * H + y) * W + x : 0;
        has[j] = (t > 0 ? TM : 0) | (t < T - 1 ? TP : 0) | (y > 0 ? UP : 0) | (x > 0 ? LEFT : 0) |
                 (x < W - 1 ? RIGHT : 0) | (y < H - 1 ? DOWN : 0) |
                 ((ox == 0 && x > 0) || (ox == bx - 1 && x < W - 1) || (oy == 0 && y > 0) ||
                          (oy == by - 1 && y < H - 1) || (ot == 0 && t > 0) || (ot == bt - 1 && t < T - 1)
                      ? OUTER : 0);
#pragma unroll
        for (int k = 0; k < K; k++) q[j][k] = C(0);
        if (in) {
            load_node(li[j], gn[j]);
            grid_dataterm_u<C, K>(gd, A.p.x, gn[j], sizeof(S) == 4, q[j]);
        }
    }
    // the nodes around the brick: the frames before and after, then the ring of every frame (its
    // corners are neighbours of no node); tile index and place in a set of its owner
    int hl[HPT], hs[HPT];
    const int face = bx * by, ring = 2 * (bx + by);
#pragma unroll
    for (int h = 0; h < HPT; h++) {
        const int u = tid + h * NT;
        int ox = 0, oy = 0, ot = 0;
        if (u < 2 * face) {
            ot = u < face ? -1 : bt;
            const int v = u < face ? u : u - face;
            ox = v % bx;
            oy = v / bx;
        } else {
            const int v = (u - 2 * face) % ring;
            ot = (u - 2 * face) / ring - 1;
            ox = v < 2 * bx ? v % bx : (v - 2 * bx < by ? -1 : bx);
            oy = v < 2 * bx ? (v < bx ? -1 : by) : (v - 2 * bx) % by;
        }
        const int x = x0 + ox, y = y0 + oy, t = t0 + ot;
        const bool in = u < 2 * face + ring * et_ && x >= 0 && x < W && y >= 0 && y < H && t >= 0 && t < T;
        hl[h] = in ? (ot + 1) * pt + (oy + 1) * py + ox + 1 : -1;
        hs[h] = 0;
        if (in) {
            const int nb = ((t / bt) * ny + y / by) * nx + x / bx;
            hs[h] = nb * brick * KS + ((t % bt) * by + y % by) * bx + x % bx;
            load_node(hl[h], (t * H + y) * W + x);
        }
    }
    __syncthreads();

    // gamma_i from gamma_{i-1} and d_{i-1} (grid_gamma_at's arithmetic)
    auto advance = [&](int at) {
        C v[K];
#pragma unroll
        for (int k = 0; k < KS; k++) v[k] = gam[k * ts + at] + beta * dir[k * ts + at];
        if (KS < K) v[K - 1] = last_row(v);
#pragma unroll
        for (int k = 0; k < K; k++) gam[k * ts + at] = v[k];
    };
    // the Laplacian at a node, the neighbours in for_neighbours' order
    auto laplacian = [&](int at, int has, const C(&g0)[K], C(&lap)[K]) {
        const C tm = has & TM ? C(1) : C(0), tp = has & TP ? C(1) : C(0);
        const C w[4] = {has & UP ? C(1) : C(0), has & LEFT ? C(1) : C(0), has & RIGHT ? C(1) : C(0),
                        has & DOWN ? C(1) : C(0)};
        const int off[4] = {-py, -1, 1, py};
#pragma unroll
        for (int k = 0; k < K; k++) {
            const C *g = gam + k * ts + at;
            lap[k] = C(2) * tm * (g0[k] - g[-pt]);
            lap[k] += C(2) * tp * (g0[k] - g[pt]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const C wm = w[i] * tm, wp = w[i] * tp;
#pragma unroll
            for (int k = 0; k < K; k++) {
                const C *g = gam + k * ts + at + off[i];
                lap[k] += w[i] * (g0[k] - g[0]);
                lap[k] += wm * (g0[k] - g[-pt]);
                lap[k] += wp * (g0[k] - g[pt]);
            }
        }
    };
    auto residual = [&](const C(&g0)[K], const C(&g)[K]) {
        C z[K];
#pragma unroll
        for (int k = 0; k < K; k++) z[k] = g0[k] - s_kkt * g[k];
        project_simplex<K, C>(z);
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++) m = nan_max(m, fabs((double)g0[k] - (double)z[k]));
        return m;
    };
    // d at a node, the last component from the others (load_dir)
    auto node_dir = [&](int at, double(&d)[K]) {
#pragma unroll
        for (int k = 0; k < KS; k++) d[k] = (double)dir[k * ts + at];
        if (KS < K) d[K - 1] = last_dir<double, K>(d);
    };

    const bool want_kkt = !A.kkt_last;  // the graph kernels form the residual in every pass
    bool fresh = first;                 // gamma_0 stands
    int e = 0;
    for (; e < A.epochs; e++) {
        double *ex = A.ex + sum_words(nwg) * e;
        double *set = A.edges + (int64_t)(e % IMG_SETS) * nwg * brick * KS;
        double *mine = set + (int64_t)wg * brick * KS;
        double *empty = A.edges + ((int64_t)((e + 2) % IMG_SETS) * nwg + wg) * brick * KS;
        double acc[NPART] = {0.0, 0.0, 0.0, 0.0, 0.0};
        // 1. gamma_i
        if (!fresh) {
#pragma unroll
            for (int j = 0; j < NPT; j++)
            {
                int at = li[j];
                asm volatile("" : "+v"(at));
                if (at >= 0) advance(at);
            }
#pragma unroll
            for (int h = 0; h < HPT; h++)
            {
                int at = hl[h];
                asm volatile("" : "+v"(at));
                if (at >= 0) advance(at);
            }
            lds_barrier();
        }
        // 2. the direction and the node sums (last iteration's marks are complete)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < NPT; j++) {
            int at = li[j], f = has[j];
            asm volatile("" : "+v"(at), "+v"(f));  // what follows from them is not kept: it would spill
            if (at < 0) continue;
            C g0[K], lap[K], g[K], y[K], p[K];
#pragma unroll
            for (int k = 0; k < K; k++) g0[k] = gam[k * ts + at];
            laplacian(at, f, g0, lap);
#pragma unroll
            for (int k = 0; k < K; k++) {
                g[k] = alpha * lap[k] + q[j][k];
                y[k] = g0[k] - a_dir * g[k];
                p[k] = y[k];
            }
            const C tau = project_simplex<K, C>(p);
            const int o = tid + j * NT;
            double ddt = 0.0, off = 0.0, fq = 0.0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                const C d = p[k] - g0[k];
                if (k < KS) {
                    dir[k * ts + at] = d;
                    if (f & OUTER) {
                        store_coherent(mine + k * brick + o, (double)d);
                        store_coherent(empty + k * brick + o, __builtin_bit_cast(double, PART_EMPTY));
                    }
                }
                ddt += (double)d * (double)d;
                const C r = tau - y[k];
                // y = tau = -inf (an overflow) gives NaN, which ends the solve, as in the graph kernels
                off += (double)(r < C(0) ? C(0) : r) * (double)g0[k];
                fq += ((double)g[k] + (double)q[j][k]) * (double)g0[k];
            }
            acc[2] += ddt + off;
            acc[3] += fq;
            if (want_kkt) acc[4] = nan_max(acc[4], residual(g0, g));
            __builtin_amdgcn_sched_barrier(0);
        }
        // 3. d_i around the brick
        {
            double v[HPT][KS];
            bool all;
            int n = 0;
            do {
                all = true;
#pragma unroll
                for (int h = 0; h < HPT; h++)
#pragma unroll
                    for (int k = 0; k < KS; k++)
                        v[h][k] = hl[h] >= 0 ? load_coherent(set + hs[h] + k * brick) : 0.0;
#pragma unroll
                for (int h = 0; h < HPT; h++)
#pragma unroll
                    for (int k = 0; k < KS; k++) all = all && published(v[h][k]);
            } while (!all && ++n < LOOP_SPIN_LIMIT);
            if (!all) A.flags[1] = 1;
#pragma unroll
            for (int h = 0; h < HPT; h++)
                if (hl[h] >= 0)
#pragma unroll
                    for (int k = 0; k < KS; k++) dir[k * ts + hl[h]] = C(v[h][k]);
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < NPT; j++) {
            int at = li[j], f = has[j];
            asm volatile("" : "+v"(at), "+v"(f));
            if (at < 0) continue;
            const double tp = f & TP ? 1.0 : 0.0;
            const double w[7] = {2.0 * tp, f & UP ? tp : 0.0, f & LEFT ? tp : 0.0, f & RIGHT ? 1.0 : 0.0,
                                 f & RIGHT ? tp : 0.0, f & DOWN ? 1.0 : 0.0, f & DOWN ? tp : 0.0};
            const int to[7] = {pt, pt - py, pt - 1, 1, pt + 1, py, pt + py};
            double d0[K];
            node_dir(at, d0);
#pragma unroll
            for (int k = 0; k < K; k++) acc[0] += d0[k] * d0[k];
#pragma unroll
            for (int i = 0; i < 7; i++) {
                double d1[K], s = 0.0;
                node_dir(at + to[i], d1);
#pragma unroll
                for (int k = 0; k < K; k++) s += (d0[k] - d1[k]) * (d0[k] - d1[k]);
                acc[1] += w[i] * s;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // 4. the sums and the step
        loop_sums<NW>(sh, acc, want_kkt, lane, wave);
        lds_barrier();
        if (wave == 0)
            loop_step(sh, want_kkt, alpha_d, (double)a_dir, sample_eps, ex, slot_ld, nwg, wg, lane, st,
                      window, A.sp, A.flags);
        lds_barrier();
        beta = uni(C(sh.b_apply));
        a_dir = uni(C(sh.a_dir));
        fresh = false;
        if (uni(sh.active) == 0) break;
    }
    // the residual of the iterate that stopped, where no iteration asked for it
    if (A.kkt_last && uni(sh.active) == 0) {
        double kkt = 0.0;
#pragma unroll
        for (int j = 0; j < NPT; j++) {
            if (li[j] < 0) continue;
            C g0[K], lap[K], g[K];
#pragma unroll
            for (int k = 0; k < K; k++) g0[k] = gam[k * ts + li[j]];
            laplacian(li[j], has[j], g0, lap);
#pragma unroll
            for (int k = 0; k < K; k++) g[k] = alpha * lap[k] + q[j][k];
            kkt = nan_max(kkt, residual(g0, g));
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
    // gamma_i (K rows, the last as complete_last_row forms it) and d_i to the launch's other buffers
    const int par = uni(sh.parity);
    S *dst = reinterpret_cast<S *>(par ? A.p.gamma1 : A.p.gamma0) + goff;
    S *dout = reinterpret_cast<S *>(par ? A.p.dir1 : A.p.dir0) + goff;
#pragma unroll
    for (int j = 0; j < NPT; j++) {
        if (li[j] < 0) continue;
        C v[K];
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = gam[k * ts + li[j]];
        if (KS < K) v[K - 1] = last_row(v);
#pragma unroll
        for (int k = 0; k < K; k++) dst[k * ld + gn[j]] = v[k];
#pragma unroll
        for (int k = 0; k < KS; k++) dout[k * ld + gn[j]] = dir[k * ts + li[j]];
    }
    if (wg == 0 && wave == 0) {
        st.parity = par;
        loop_put_state(A.state[0], A.sp.m, lane, st, window);
        loop_put_state(*A.out, A.sp.m, lane, st, window);
        if (lane == 0) A.flags[0] = st.active;
    }
}

}  // namespace pasc
