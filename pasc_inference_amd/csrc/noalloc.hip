// The theta step without device allocations (pasc_theta_update_noalloc).
//
// pasc_theta_update keeps its workgroups' partial sums in the engine's scratch buffer, which grows
// by hipMalloc when it is too small.  Callers that cannot allocate (code under HIP graph capture,
// tight serving loops) use this variant instead: the same kernels with the partials in
// `scratch`, a file-scope device array of NOALLOC_SCRATCH_DOUBLES doubles (4 MiB on every device
// the library runs on, held until the process ends), so the two give bit-identical theta.
//
// Every call on a device shares that device's array: calls that overlap on one device race.
// The array is addressed through the pointer hipGetSymbolAddress returned for the device
// (noalloc_init, run by pasc_ctx_create with the device current); the array's name is a
// host-side stand-in that no host code may pass to a kernel.
#include <hip/hip_runtime.h>

#include <mutex>

#include "util_kernels.h"

namespace pasc {

constexpr size_t NOALLOC_SCRATCH_DOUBLES = (size_t)1 << 19;  // 4 MiB
constexpr int NOALLOC_MAX_DEVICES = 64;

static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];

static std::mutex g_scratch_mu;
static double *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// Device address of `scratch` on `device` (the caller made it current).  Once per device.
int noalloc_init(int device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES)
        return fail(PASC_ERR_ARG, "noalloc: device %d beyond %d", device, NOALLOC_MAX_DEVICES);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return PASC_OK;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return fail(PASC_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", device,
                    hipGetErrorString(e));
    g_scratch_ptr[device] = (double *)ptr;
    return PASC_OK;
}

// Largest number of steps the call takes for K clusters and xdim channels: a row of partials per 256
// steps, less one, in the scratch.  (The sums take at most READ_BLOCKS rows whatever the steps; the
// limit stands as the interface states it.)
int64_t noalloc_theta_max_T(int K, int xdim) {
    const int64_t nv = (int64_t)K * (1 + xdim);
    const int64_t blocks = (int64_t)NOALLOC_SCRATCH_DOUBLES / nv - 1;
    return blocks * 256;
}

// The theta step of rows_theta with the partials in the static scratch: gamma rows g (type f32
// or FP64) described by d, data rows x of stride d.ld; theta_out receives theta[k*xdim + c].
int rows_theta_noalloc(Engine &e, const void *g, bool f32, const InstDesc &d, const double *x,
                       double *theta_out) {
    const int device = e.ctx->device;
    if (device < 0 || device >= NOALLOC_MAX_DEVICES || !g_scratch_ptr[device])
        return fail(PASC_ERR_STATE, "theta_update_noalloc: the static scratch of device %d was "
                                    "not set up (pasc_ctx_create does that)", device);
    if (d.T > noalloc_theta_max_T(d.K, d.xdim))
        return fail(PASC_ERR_ARG, "theta_update_noalloc: T*R = %lld exceeds %lld, the most the "
                                  "call takes at K = %d, xdim = %d",
                    (long long)d.T, (long long)noalloc_theta_max_T(d.K, d.xdim), d.K, d.xdim);
    static_assert(NOALLOC_SCRATCH_DOUBLES >= (size_t)READ_BLOCKS * PASC_MAX_K * 4, "the partials fit");
    return theta_from_rows(e, g, f32, d, x, g_scratch_ptr[device], theta_out);
}

}  // namespace pasc
