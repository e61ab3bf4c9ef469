// The adjoint of a 1-D problem in one persistent launch: the right-hand side, every CG step of
// (P A P) lambda = P dJ/dgamma and the gradient's sums, with r, p and lambda on chip.
//
// A CG step as kernels reads and writes 10 vectors (240 MB at T = 1e6, K = 3) in four launches and
// took 55 us there, 26 + 20 us of it for the vectors at the rate of the last-level cache.  Here a
// wave owns 64 x CH consecutive steps, r and p in registers and lambda in LDS, so a step costs
// its arithmetic and two exchanges of one sum between the workgroups (exchange.h; see
// loop_kernels.h for the scheme and the cooperative launch): 7.4 us, about 2 us of it each
// exchange (10 us with the sums in one copy, barriers that waited for the edges' stores too and
// lambda advanced before r'r was published).  The neighbouring waves' edge values
// of p are not exchanged: each wave keeps copies and advances them with the edges of r, which
// travel with r'r.
// A lane holds up to 8 steps for K <= 4 (r, p and q: 48 doubles at K = 3 and 8 steps, within the
// 256 registers of 8 waves a workgroup) and up to 4 for larger K: 1.05 million steps (0.52) on 256
// CUs.  Shorter series take fewer steps a lane and fewer waves while every wave still has a CU to
// itself or shares it with seven others.
#pragma once

#include "exchange.h"
#include "spg_kernels.h"

namespace pasc {

struct AdjLoopArgs {
    const double *gam;      // gamma* rows (stride ld)
    const double *x;        // data row
    const uint8_t *mask;    // held-out steps (1 = in the loss)
    const uint8_t *qmask;   // steps without a data term in the QP, or null
    int64_t T, ld;
    double alpha, bscale, tol2;
    double theta[PASC_MAX_K];
    double *save;           // r, p, lambda between launches: 3 x [K][ld]
    double *save_rr;        // r'r and the step count between launches
    double *out;            // pinned: J, lambda' A gamma, direct + implicit dJ/dtheta_k
    int32_t *flags;         // pinned: [0] 1 while CG has not stopped, [1] a wait ran out, [2] steps
    double *ex;             // exchange area
    int32_t epochs;         // CG steps of this launch at most
    int32_t maxit;
    int32_t resume;         // 1: r, p and lambda come from save
};

constexpr int adj_chunk(int K) { return K <= 4 ? 8 : 4; }  // steps of a lane at most
// exchange area: the opening and closing sums, then per CG step two sums and the edges of r
template <int K>
__host__ __device__ constexpr int64_t adj_open_words(int nwg) {
    return (int64_t)slot_stride(nwg) * (2 + K) * 2 + (int64_t)nwg * 2 * K;
}
template <int K>
__host__ __device__ constexpr int64_t adj_epoch_words(int nwg) {
    return (int64_t)slot_stride(nwg) * 2 * SUM_COPIES + (int64_t)nwg * 2 * K;
}

// P applied to the K values of one step (free set in the low K bits of fr)
template <int K>
__device__ __forceinline__ void face_project(double (&v)[K], unsigned fr) {
    double s = 0.0;
    int nf = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const bool f = (fr >> k) & 1u;
        s += f ? v[k] : 0.0;
        nf += f ? 1 : 0;
    }
    const double m = s * recip_small<double, K>(nf);
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = ((fr >> k) & 1u) && nf > 1 ? v[k] - m : 0.0;
}

template <int K, int CH, int NW>
__global__ __launch_bounds__(NW *WAVE) void adj_loop(AdjLoopArgs A) {
    extern __shared__ __attribute__((aligned(16))) double lam[];  // [K][NW * WAVE * CH]
    __shared__ double red[2 + K][NW];
    __shared__ double redge[2][NW + 2][2][K];  // r at a wave's first and last step, by CG parity
    __shared__ double bc[2];                   // step (or b), stop
    const int nwg = gridDim.x, wg = blockIdx.x, sld = slot_stride(nwg);
    const int lane = threadIdx.x & (WAVE - 1), wave = uni((int32_t)(threadIdx.x / WAVE));
    const int64_t T = A.T, ld = A.ld;
    const int64_t t0 = ((int64_t)wg * NW + wave) * (WAVE * CH) + (int64_t)lane * CH;
    double *my_lam = lam + (wave * WAVE + lane) * CH;
    constexpr int LROW = NW * WAVE * CH;
    int32_t *lost = A.flags + 1;

    // V sums over the workgroup in red[v][0 .. NW), published as rows of `row`
    auto publish = [&](double *row, int nv) {
        __syncthreads();
        if (wave == 0) {
            for (int v = 0; v < nv; v++) {
                const double s = wave_sum_all(lane < NW ? red[v][lane] : 0.0);
                if (lane == 0) store_coherent(row + (int64_t)v * sld + wg, s);
            }
        }
    };
    // the sum of a CG step: in SUM_COPIES rows, each workgroup reading one (see exchange.h)
    auto publish_step = [&](double *rows) {
        lds_barrier();
        if (wave == 0) {
            const double s = wave_sum_all(lane < NW ? red[0][lane] : 0.0);
            if (lane < SUM_COPIES) store_coherent(rows + (int64_t)lane * sld + wg, s);
        }
    };
    const int64_t copy = (int64_t)(wg % SUM_COPIES) * sld;
    // the wave's edge steps of v to LDS and, at the workgroup's ends, to the exchange area
    auto put_edges = [&](int par, const double(&v)[K][CH], double *ex_edges) {
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                redge[par][wave + 1][0][k] = v[k][0];
                if (wave == 0 && wg > 0) store_coherent(ex_edges + ((int64_t)wg * 2) * K + k, v[k][0]);
            }
        }
        if (lane == WAVE - 1) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                redge[par][wave + 1][1][k] = v[k][CH - 1];
                if (wave == NW - 1 && wg < nwg - 1)
                    store_coherent(ex_edges + ((int64_t)wg * 2 + 1) * K + k, v[k][CH - 1]);
            }
        }
    };
    // the neighbouring workgroups' edges into LDS (by one wave; 0 past the series)
    auto get_edges = [&](int par, const double *ex_edges) {
        if (lane >= 2 * K) return;
        const int side = lane / K, k = lane - side * K;  // 0: from the left, 1: from the right
        const int nb = side == 0 ? wg - 1 : wg + 1;
        const double v = nb < 0 || nb >= nwg
                             ? 0.0
                             : await_value(ex_edges + ((int64_t)nb * 2 + (side ^ 1)) * K + k, lost);
        redge[par][side == 0 ? 0 : NW + 1][side ^ 1][k] = v;
    };

    double r[K][CH], p[K][CH], pl[K], pr[K];
    unsigned fr = 0;  // free set, K bits a step
    bool held[CH];
    {
        double g[K][CH], X[CH], sums[2 + K];
#pragma unroll
        for (int v = 0; v < 2 + K; v++) sums[v] = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++) load_chunk<double, double, CH>(A.gam + k * ld, t0, T, ld, g[k]);
        load_chunk<double, double, CH>(A.x, t0, T, ld, X);
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const bool in = t0 + c < T;
            held[c] = in && A.mask[in ? t0 + c : 0] != 0;
            double rec = 0.0, dj[K];
            unsigned f = 0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                f |= g[k][c] > FREE_EPS ? 1u << k : 0u;
                rec += A.theta[k] * g[k][c];
            }
            fr |= f << (c * K);
            const double res = held[c] ? X[c] - rec : 0.0;
            sums[0] += res * res;
#pragma unroll
            for (int k = 0; k < K; k++) {
                dj[k] = -2.0 * res * A.theta[k];
                sums[2 + k] += -2.0 * res * g[k][c];
            }
            face_project<K>(dj, f);
#pragma unroll
            for (int k = 0; k < K; k++) {
                r[k][c] = dj[k];
                sums[1] += dj[k] * dj[k];
            }
        }
#pragma unroll
        for (int v = 0; v < 2 + K; v++) {
            const double s = wave_sum_all(sums[v]);
            if (lane == 0) red[v][wave] = s;
        }
    }
    double *open = A.ex, *close = A.ex + (int64_t)sld * (2 + K);
    double *open_edges = close + (int64_t)sld * (2 + K);
    if (A.resume) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            load_chunk<double, double, CH>(A.save + k * ld, t0, T, ld, r[k]);
            load_chunk<double, double, CH>(A.save + (K + k) * ld, t0, T, ld, p[k]);
            double l[CH];
            load_chunk<double, double, CH>(A.save + (2 * K + k) * ld, t0, T, ld, l);
#pragma unroll
            for (int c = 0; c < CH; c++) my_lam[k * LROW + c] = l[c];
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < CH; c++) {
                p[k][c] = r[k][c];
                my_lam[k * LROW + c] = 0.0;
            }
    }
    put_edges(0, p, open_edges);
    publish(open, 2 + K);
    if (wave == NW - 1) get_edges(0, open_edges);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        pl[k] = redge[0][wave][1][k];
        pr[k] = redge[0][wave + 2][0][k];
    }
    // CG scalars, in wave 0
    double rr = 0.0, rr0 = 0.0, loss = 0.0, direct[K];
    int it = 0;
    const int maxit = A.maxit;
    bool done = false;
    if (wave == 0) {
        loss = await_sum(open, nwg, lane, lost);
        rr0 = await_sum(open + sld, nwg, lane, lost);
#pragma unroll
        for (int k = 0; k < K; k++)
            direct[k] = await_sum(open + (int64_t)(2 + k) * sld, nwg, lane, lost);
        rr = A.resume ? A.save_rr[0] : rr0;
        it = A.resume ? (int)A.save_rr[1] : 0;
        done = !(it < maxit && rr > A.tol2 * rr0 && rr > 0.0);
        if (lane == 0) bc[1] = done ? 1.0 : 0.0;
    }
    __syncthreads();
    bool stop = bc[1] != 0.0;

    for (int e = 0; e < A.epochs && !stop; e++) {
        double *ex = A.ex + adj_open_words<K>(nwg) + adj_epoch_words<K>(nwg) * e;
        double *ex_r = ex + SUM_COPIES * (int64_t)sld, *ex_edges = ex_r + SUM_COPIES * (int64_t)sld;
        const int par = e & 1;
        // q = P A p and p'q
        double q[K][CH], pq = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++) {
            double left = dpp_shift<DPP_WAVE_SHR1>(p[k][CH - 1]);
            double right = dpp_shift<DPP_WAVE_SHL1>(p[k][0]);
            left = lane == 0 ? pl[k] : left;
            right = lane == WAVE - 1 ? pr[k] : right;
#pragma unroll
            for (int c = 0; c < CH; c++) {
                const int64_t t = t0 + c;
                const double vm = c > 0 ? p[k][c - 1] : left, vp = c < CH - 1 ? p[k][c + 1] : right;
                double l = t > 0 ? 2.0 * (p[k][c] - vm) : 0.0;
                l += t < T - 1 ? 2.0 * (p[k][c] - vp) : 0.0;
                q[k][c] = A.alpha * l;
            }
        }
#pragma unroll
        for (int c = 0; c < CH; c++) {
            double w[K];
#pragma unroll
            for (int k = 0; k < K; k++) w[k] = q[k][c];
            face_project<K>(w, fr >> (c * K));  // (no step past the end is free)
#pragma unroll
            for (int k = 0; k < K; k++) {
                q[k][c] = w[k];
                pq += p[k][c] * w[k];
            }
        }
        pq = wave_sum_all(pq);
        if (lane == 0) red[0][wave] = pq;
        publish_step(ex);
        if (wave == 0) {
            pq = await_sum(ex + copy, nwg, lane, lost);
            if (lane == 0) {
                bc[0] = rr / pq;
                bc[1] = pq > 0.0 ? 0.0 : 1.0;  // p in the null space of P A P: the system is solved
            }
        }
        lds_barrier();
        const double step = bc[0];
        stop = bc[1] != 0.0;
        if (stop) break;
        // r -= step q, r'r
        double rn = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < CH; c++) {
                r[k][c] -= step * q[k][c];
                rn += r[k][c] * r[k][c];
            }
        put_edges(par ^ 1, r, ex_edges);
        rn = wave_sum_all(rn);
        if (lane == 0) red[0][wave] = rn;
        publish_step(ex_r);
        // lambda += step p while the sums travel
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < CH; c++) my_lam[k * LROW + c] += step * p[k][c];
        if (wave == NW - 1) get_edges(par ^ 1, ex_edges);
        if (wave == 0) {
            rn = await_sum(ex_r + copy, nwg, lane, lost);
            const double b = rn / rr;
            rr = rn;
            it++;
            done = !(it < maxit && rn > A.tol2 * rr0 && rn > 0.0);
            if (lane == 0) {
                bc[0] = b;
                bc[1] = done ? 1.0 : 0.0;
            }
        }
        lds_barrier();
        const double b = bc[0];
        stop = bc[1] != 0.0;
#pragma unroll
        for (int k = 0; k < K; k++) {
#pragma unroll
            for (int c = 0; c < CH; c++) p[k][c] = r[k][c] + b * p[k][c];
            pl[k] = redge[par ^ 1][wave][1][k] + b * pl[k];
            pr[k] = redge[par ^ 1][wave + 2][0][k] + b * pr[k];
        }
    }
    if (!stop) {
        // more steps than this launch holds: the state for the next one
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < CH; c++)
                if (t0 + c < T) {
                    A.save[k * ld + t0 + c] = r[k][c];
                    A.save[(K + k) * ld + t0 + c] = p[k][c];
                    A.save[(2 * K + k) * ld + t0 + c] = my_lam[k * LROW + c];
                }
        if (wg == 0 && wave == 0 && lane == 0) {
            A.save_rr[0] = rr;
            A.save_rr[1] = (double)it;
            A.flags[0] = 1;
        }
        return;
    }
    // lambda' A gamma and the implicit part of dJ/dtheta
    {
        double sums[1 + K], X[CH];
#pragma unroll
        for (int v = 0; v < 1 + K; v++) sums[v] = 0.0;
        load_chunk<double, double, CH>(A.x, t0, T, ld, X);
#pragma unroll
        for (int k = 0; k < K; k++) {
            double g[CH];
            const double *row = A.gam + k * ld;
            load_chunk<double, double, CH>(row, t0, T, ld, g);
            const double left = t0 > 0 && t0 - 1 < T ? row[t0 - 1] : 0.0;
            const double right = t0 + CH < T ? row[t0 + CH] : 0.0;
#pragma unroll
            for (int c = 0; c < CH; c++) {
                const int64_t t = t0 + c;
                const double vm = c > 0 ? g[c - 1] : left, vp = c < CH - 1 ? g[c + 1] : right;
                double l = t > 0 ? 2.0 * (g[c] - vm) : 0.0;
                l += t < T - 1 ? 2.0 * (g[c] - vp) : 0.0;
                const double lk = t < T ? my_lam[k * LROW + c] : 0.0;
                sums[0] += lk * A.alpha * l;
                // the data term of a step without one does not depend on theta
                const bool data = t < T && !(A.qmask && A.qmask[t] != 0);
                sums[1 + k] += data ? lk * 2.0 * (X[c] - A.theta[k]) * A.bscale : 0.0;
            }
        }
#pragma unroll
        for (int v = 0; v < 1 + K; v++) {
            const double s = wave_sum_all(sums[v]);
            if (lane == 0) red[v][wave] = s;
        }
        publish(close, 1 + K);
        if (wg == 0 && wave == 0) {
            const double v0 = await_sum(close, nwg, lane, lost);
            double dth[K];
#pragma unroll
            for (int k = 0; k < K; k++)
                dth[k] = direct[k] +
                         await_sum(close + (int64_t)(1 + k) * sld, nwg, lane, lost);
            if (lane == 0) {
                A.out[0] = loss;
                A.out[1] = v0;
#pragma unroll
                for (int k = 0; k < K; k++) A.out[2 + k] = dth[k];
                A.flags[0] = 0;
                A.flags[2] = it;
            }
        }
    }
}

}  // namespace pasc
