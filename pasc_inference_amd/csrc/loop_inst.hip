// Instantiations of the persistent 1-D loop for one storage type (PASS_S) and one workgroup size
// (LOOP_NW waves).
#include "loop_kernels.h"

#if !defined(PASS_S) || !defined(LOOP_NW)
#error "PASS_S (float or double) and LOOP_NW (waves per workgroup) must be defined"
#endif

#define PASC_CAT3_(a, b, c) a##b##c
#define PASC_CAT3(a, b, c) PASC_CAT3_(a, b, c)
#define LOOP_FN PASC_CAT3(launch_loop_1d_, PASS_S, PASC_CAT3(_, LOOP_NW, _))

namespace pasc {

template <int K, int CH>
static int launch_kc(const LoopArgs &a, int nwg, hipStream_t s) {
    if constexpr (loop_has_chunk(sizeof(PASS_S) == 8, K, CH)) {
        using L = LoopShape<PASS_S, K, CH>;
        const void *fn = reinterpret_cast<const void *>(spg_loop_1d<PASS_S, PASS_S, K, CH, LOOP_NW>);
        const size_t lds = L::lds_bytes(a.tpw);
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return PASC_ERR_HIP;
        LoopArgs args = a;
        void *params[] = {&args};
        return hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(LOOP_NW * WAVE), params,
                                          (unsigned)lds, s) == hipSuccess
                   ? PASC_OK
                   : PASC_ERR_HIP;
    }
    return PASC_ERR_HIP;
}

template <int K>
static int launch_k(const LoopArgs &a, int nwg, int chunk, hipStream_t s) {
    return chunk == 2 ? launch_kc<K, 2>(a, nwg, s) : launch_kc<K, 4>(a, nwg, s);
}

// PASC_ERR_HIP (without a message): the launch was refused, the caller runs the tiled passes
int LOOP_FN(int K, const LoopArgs &a, int nwg, int chunk, hipStream_t s) {
    switch (K) {
        case 1: return launch_k<1>(a, nwg, chunk, s);
        case 2: return launch_k<2>(a, nwg, chunk, s);
        case 3: return launch_k<3>(a, nwg, chunk, s);
        case 4: return launch_k<4>(a, nwg, chunk, s);
        case 5: return launch_k<5>(a, nwg, chunk, s);
        case 6: return launch_k<6>(a, nwg, chunk, s);
        case 7: return launch_k<7>(a, nwg, chunk, s);
        case 8: return launch_k<8>(a, nwg, chunk, s);
    }
    return PASC_ERR_HIP;
}

}  // namespace pasc
