// Host <-> device transfers of row-major state (gamma, explicit linear terms, data) in the
// layouts of the C boundary.
//
// The caller's array is in the boundary's layout (interleaved or one row after another, FP64);
// the device keeps padded rows of the problem's type.  A kernel does the change of layout and
// type and reads or writes pinned host memory directly (48 - 55 GB/s in both directions, as fast
// as the copy engine and without a device buffer in between); host threads move the pinned
// pieces from and to the caller's pages.  240 MB (T = 1e7, K = 3) took 86 ms down and 73 ms up
// when one host thread did the layout around a pageable copy; in 4 MiB pieces over 8 threads it
// takes 5 ms, of which the link needs 4.3.  One thread would be bound by its page faults and
// copies (23 ms).  Up to one piece, a single kernel moves the whole transfer and the threads share
// the host copy (1.4 MB into fresh pages: 150 us by one thread, 75 by several).  A few rows
// go by the copy engine (small_transfer).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <vector>

#include "device_common.h"
#include "team.h"

namespace pasc {

// Element i of the boundary's array: row (k) and column (t) of the device rows.
__device__ __forceinline__ void boundary_index(int64_t i, int64_t T, int K, int interleaved, int64_t &t,
                                               int &k) {
    if (interleaved) {
        t = i / K;
        k = (int)(i - t * K);
    } else {
        k = (int)(i / T);
        t = i - (int64_t)k * T;
    }
}

template <typename S>
__global__ __launch_bounds__(256) void rows_pack(const S *rows, int64_t T, int64_t ld, int K,
                                                 int interleaved, int64_t i0, int64_t n,
                                                 double *out) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int64_t t;
        int k;
        boundary_index(i0 + i, T, K, interleaved, t, k);
        out[i] = (double)rows[k * ld + t];
    }
}

template <typename S>
__global__ __launch_bounds__(256) void rows_unpack(const double *in, int64_t T, int64_t ld, int K,
                                                   int interleaved, int64_t i0, int64_t n,
                                                   S *rows) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int64_t t;
        int k;
        boundary_index(i0 + i, T, K, interleaved, t, k);
        rows[k * ld + t] = S(in[i]);
    }
}

// Pinned pieces of one device, shared by its contexts: at most SLOTS of SLOT_BYTES, allocated
// when first needed and freed with the device's last context.  A transfer holds the slots it
// works on and waits for none but its first, so transfers of several threads share them.
struct Slot {
    double *p = nullptr;
    hipEvent_t ev = nullptr;
};
constexpr int SLOTS = 8;
constexpr size_t SLOT_BYTES = (size_t)4 << 20;
constexpr int POOL_DEVICES = 64;
constexpr size_t COPY_PIECE = (size_t)128 << 10;  // share of a host copy worth another thread

struct SlotPool {
    std::mutex mu;
    std::condition_variable cv;
    std::vector<Slot> idle;
    int allocated = 0;
    int users = 0;

    // a slot, or none when all are taken and wait is false
    hipError_t take(bool wait, Slot &s) {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            if (!idle.empty()) {
                s = idle.back();
                idle.pop_back();
                return hipSuccess;
            }
            if (allocated < SLOTS) {
                Slot n;
                hipError_t e = hipHostMalloc((void **)&n.p, SLOT_BYTES, hipHostMallocDefault);
                if (e != hipSuccess) return e;
                e = hipEventCreateWithFlags(&n.ev, hipEventDisableTiming);
                if (e != hipSuccess) {
                    (void)hipHostFree(n.p);
                    return e;
                }
                allocated++;
                s = n;
                return hipSuccess;
            }
            if (!wait) return hipErrorNotReady;
            cv.wait(lk);
        }
    }
    void give(const Slot &s) {
        {
            std::lock_guard<std::mutex> lk(mu);
            idle.push_back(s);
        }
        cv.notify_one();
    }
};

static SlotPool *const g_pool = new SlotPool[POOL_DEVICES];

static_assert(Team::MOST == SLOTS - 1, "a slot for the calling thread and one for every helper");

// never destroyed: parked threads end with the process when a context is still open then
static Team &g_team = *new Team;

int staging_open(int device) {
    if (device < 0 || device >= POOL_DEVICES)
        return fail(PASC_ERR_ARG, "staging: device %d beyond %d", device, POOL_DEVICES);
    SlotPool &p = g_pool[device];
    g_team.open();
    std::lock_guard<std::mutex> lk(p.mu);
    p.idle.reserve(SLOTS);
    p.users++;
    return PASC_OK;
}

void staging_close(int device) {
    if (device < 0 || device >= POOL_DEVICES) return;
    g_team.close();
    SlotPool &p = g_pool[device];
    std::lock_guard<std::mutex> lk(p.mu);
    if (--p.users > 0) return;
    for (auto &s : p.idle) {
        (void)hipEventDestroy(s.ev);
        (void)hipHostFree(s.p);
    }
    p.allocated -= (int)p.idle.size();
    p.idle.clear();
}

// memcpy by several threads
static void team_copy(void *dst, const void *src, size_t bytes) {
    const int n = (int)std::min<size_t>((size_t)Team::helpers(), bytes / COPY_PIECE);
    if (n < 1) {
        std::memcpy(dst, src, bytes);
        return;
    }
    const size_t share = (bytes / (n + 1) + 4095) / 4096 * 4096;
    std::atomic<size_t> next{0};
    g_team.run(n, [&]() {
        for (size_t i = next.fetch_add(share); i < bytes; i = next.fetch_add(share))
            std::memcpy((char *)dst + i, (const char *)src + i, std::min(share, bytes - i));
    });
}

// One transfer: pieces of `piece` elements, taken in turn by the calling thread and its helpers.
struct Transfer {
    int device;
    hipStream_t stream;
    bool to_host, single;
    char *host;
    size_t esize;
    int64_t total, piece;
    const PieceLaunch *launch;
    std::atomic<int64_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    std::atomic<bool> caller{true};

    void copy(void *dst, const void *src, size_t bytes) {
        if (single) team_copy(dst, src, bytes);
        else std::memcpy(dst, src, bytes);
    }

    hipError_t one(const Slot &s, int64_t i0, int64_t n) {
        if (!to_host) copy(s.p, host + (size_t)i0 * esize, (size_t)n * esize);
        (*launch)(stream, i0, n, s.p);
        hipError_t e;
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = hipEventRecord(s.ev, stream)) != hipSuccess) return e;
        if ((e = hipEventSynchronize(s.ev)) != hipSuccess) return e;
        if (to_host) copy(host + (size_t)i0 * esize, s.p, (size_t)n * esize);
        return hipSuccess;
    }

    // The first to come waits for a slot; the others leave when there is none.
    void work() {
        const bool first = caller.exchange(false);
        hipError_t e = hipSetDevice(device);
        Slot s;
        if (e == hipSuccess) {
            e = g_pool[device].take(first, s);
            if (!first && e != hipSuccess) return;  // the others do the work
        }
        if (e == hipSuccess) {
            for (int64_t i = next.fetch_add(piece); i < total && error.load() == (int)hipSuccess;
                 i = next.fetch_add(piece)) {
                e = one(s, i, std::min(piece, total - i));
                if (e != hipSuccess) break;
            }
            g_pool[device].give(s);
        }
        if (e != hipSuccess) {
            int none = (int)hipSuccess;
            error.compare_exchange_strong(none, (int)e);
        }
    }
};

int with_input(Ctx *ctx, const void *host, size_t bytes, const std::function<void(const void *)> &launch) {
    if (bytes > SLOT_BYTES) return fail(PASC_ERR_ARG, "with_input: %zu bytes", bytes);
    SlotPool &pool = g_pool[ctx->device];
    Slot s;
    hipError_t e = pool.take(true, s);
    if (e == hipSuccess) {
        std::memcpy(s.p, host, bytes);
        launch(s.p);
        e = hipGetLastError();
        const hipError_t w = hipStreamSynchronize((hipStream_t)ctx->stream);
        if (e == hipSuccess) e = w;
        pool.give(s);
    }
    return e == hipSuccess ? PASC_OK : fail(PASC_ERR_HIP, "host to device: %s", hipGetErrorString(e));
}

// Whole slots, or an eighth of a transfer that would fill only a few.
int64_t staged_piece(size_t esize, int64_t total) {
    const int64_t slot = (int64_t)(SLOT_BYTES / esize);
    if (total <= slot) return slot;
    const int64_t unit = (int64_t)(COPY_PIECE / esize), share = (total + SLOTS - 1) / SLOTS;
    return std::min(slot, std::max(8 * unit, (share + unit - 1) / unit * unit));
}

int staged_transfer(Ctx *ctx, bool to_host, void *host, size_t esize, int64_t total,
                    const PieceLaunch &launch) {
    if (total <= 0) return PASC_OK;
    Transfer t;
    t.device = ctx->device;
    t.stream = (hipStream_t)ctx->stream;
    t.to_host = to_host;
    t.host = (char *)host;
    t.esize = esize;
    t.total = total;
    t.launch = &launch;
    t.piece = staged_piece(esize, total);
    t.single = total <= t.piece;
    const int64_t pieces = (total + t.piece - 1) / t.piece;
    g_team.run((int)std::min<int64_t>(Team::helpers(), pieces - 1), [&t]() { t.work(); });
    const hipError_t e = (hipError_t)t.error.load();
    if (e != hipSuccess)
        return fail(PASC_ERR_HIP, "%s transfer: %s", to_host ? "device to host" : "host to device",
                    hipGetErrorString(e));
    return PASC_OK;
}

static unsigned piece_blocks(int64_t n) { return (unsigned)std::min<int64_t>((n + 255) / 256, 1024); }

// Transfers of a few rows: the rows as they lie by the copy engine, the change of layout and type on
// this thread.  us of a whole call, FP64, K = 3, interleaved, against a kernel, its event and parked
// threads: up 24 KB 10.7 / 17.9, 240 KB 16.7 / 29, 1 MB 44 / 60; down into pages of an earlier call
// 10.8 / 17.4, 21.4 / 30, 50 / 65.  Down into fresh pages the threads share the page faults: 240 KB
// 41 / 47 - 66, 375 KB 66 / 75, 470 KB 83 / 85 (one row after another 96 / 86), 940 KB 167 / 153.
constexpr size_t SMALL_UP = (size_t)1 << 20, SMALL_DOWN = (size_t)400 << 10;

// rows of T values to and from the interleaved order (K known: the rows are walked together)
template <int K, typename S>
static void weave(const S *rows, int64_t T, int64_t ld, double *host) {
    for (int64_t t = 0; t < T; t++)
        for (int k = 0; k < K; k++) host[t * K + k] = (double)rows[k * ld + t];
}
template <int K, typename S>
static void unweave(const double *host, int64_t T, int64_t ld, S *rows) {
    for (int64_t t = 0; t < T; t++)
        for (int k = 0; k < K; k++) rows[k * ld + t] = S(host[t * K + k]);
}

template <typename S>
static void rows_to_boundary(const S *rows, int64_t T, int64_t ld, int K, double *host, bool interleaved) {
    switch (interleaved ? K : 1) {
        case 2: return weave<2>(rows, T, ld, host);
        case 3: return weave<3>(rows, T, ld, host);
        case 4: return weave<4>(rows, T, ld, host);
        case 5: return weave<5>(rows, T, ld, host);
        case 6: return weave<6>(rows, T, ld, host);
        case 7: return weave<7>(rows, T, ld, host);
        case 8: return weave<8>(rows, T, ld, host);
    }
    for (int k = 0; k < K; k++) std::copy(rows + k * ld, rows + k * ld + T, host + k * T);
}

template <typename S>
static void boundary_to_rows(const double *host, int64_t T, int64_t ld, int K, S *rows, bool interleaved) {
    for (int k = 0; k < K; k++) std::fill(rows + k * ld + T, rows + (k + 1) * ld, S(0));  // as allocated
    switch (interleaved ? K : 1) {
        case 2: return unweave<2>(host, T, ld, rows);
        case 3: return unweave<3>(host, T, ld, rows);
        case 4: return unweave<4>(host, T, ld, rows);
        case 5: return unweave<5>(host, T, ld, rows);
        case 6: return unweave<6>(host, T, ld, rows);
        case 7: return unweave<7>(host, T, ld, rows);
        case 8: return unweave<8>(host, T, ld, rows);
    }
    for (int k = 0; k < K; k++)
        for (int64_t t = 0; t < T; t++) rows[k * ld + t] = S(host[k * T + t]);
}
static_assert(PASC_MAX_K == 8, "a case for every K");

static int small_transfer(Ctx *ctx, bool to_host, void *rows, bool f32, int64_t T, int64_t ld, int K,
                          double *host, bool interleaved) {
    const size_t bytes = (f32 ? 4 : 8) * (size_t)ld * K;
    SlotPool &pool = g_pool[ctx->device];
    hipStream_t stream = (hipStream_t)ctx->stream;
    Slot s;
    hipError_t e = pool.take(true, s);
    if (e == hipSuccess) {
        if (!to_host) {
            if (f32) boundary_to_rows(host, T, ld, K, (float *)s.p, interleaved);
            else boundary_to_rows(host, T, ld, K, s.p, interleaved);
        }
        e = hipMemcpyAsync(to_host ? (void *)s.p : rows, to_host ? rows : (void *)s.p, bytes,
                           to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e == hipSuccess && to_host) {
            if (f32) rows_to_boundary((const float *)s.p, T, ld, K, host, interleaved);
            else rows_to_boundary((const double *)s.p, T, ld, K, host, interleaved);
        }
        pool.give(s);
    }
    if (e != hipSuccess)
        return fail(PASC_ERR_HIP, "%s transfer: %s", to_host ? "device to host" : "host to device",
                    hipGetErrorString(e));
    return PASC_OK;
}

int rows_to_host(Ctx *ctx, const void *rows, bool f32, int64_t T, int64_t ld, int K, double *host,
                 bool interleaved) {
    if (sizeof(double) * (size_t)ld * K <= SMALL_DOWN)
        return small_transfer(ctx, true, const_cast<void *>(rows), f32, T, ld, K, host, interleaved);
    const int il = interleaved ? 1 : 0;
    return staged_transfer(
        ctx, true, host, sizeof(double), T * K, [=](hipStream_t s, int64_t i0, int64_t n, void *p) {
            if (f32)
                hipLaunchKernelGGL(rows_pack<float>, dim3(piece_blocks(n)), dim3(256), 0, s,
                                   (const float *)rows, T, ld, K, il, i0, n, (double *)p);
            else
                hipLaunchKernelGGL(rows_pack<double>, dim3(piece_blocks(n)), dim3(256), 0, s,
                                   (const double *)rows, T, ld, K, il, i0, n, (double *)p);
        });
}

int rows_from_host(Ctx *ctx, const double *host, bool interleaved, void *rows, bool f32,
                   int64_t T, int64_t ld, int K) {
    if (sizeof(double) * (size_t)ld * K <= SMALL_UP)
        return small_transfer(ctx, false, rows, f32, T, ld, K, const_cast<double *>(host), interleaved);
    const int il = interleaved ? 1 : 0;
    return staged_transfer(
        ctx, false, const_cast<double *>(host), sizeof(double), T * K,
        [=](hipStream_t s, int64_t i0, int64_t n, void *p) {
            if (f32)
                hipLaunchKernelGGL(rows_unpack<float>, dim3(piece_blocks(n)), dim3(256), 0, s,
                                   (const double *)p, T, ld, K, il, i0, n, (float *)rows);
            else
                hipLaunchKernelGGL(rows_unpack<double>, dim3(piece_blocks(n)), dim3(256), 0, s,
                                   (const double *)p, T, ld, K, il, i0, n, (double *)rows);
        });
}

}  // namespace pasc
