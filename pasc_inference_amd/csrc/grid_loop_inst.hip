// Instantiations of the persistent loop of spatio-temporal grids for one storage type (PASS_S).
#include "grid_loop.h"

#ifndef PASS_S
#error "PASS_S (float or double) must be defined"
#endif

#define PASC_CAT2_(a, b) a##b
#define PASC_CAT2(a, b) PASC_CAT2_(a, b)
#define LOOP_FN PASC_CAT2(launch_grid_loop_, PASS_S)

namespace pasc {

template <int K, int NPT>
static int launch_kn(const GridLoopArgs &a, int nwg, hipStream_t s) {
    const size_t lds = grid_loop_lds<PASS_S>(K);
    const void *fn = reinterpret_cast<const void *>(grid_loop<PASS_S, K, NPT>);
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return PASC_ERR_HIP;
    GridLoopArgs args = a;
    void *params[] = {&args};
    return hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(GRID_LOOP_NT), params, (unsigned)lds, s) ==
                   hipSuccess
               ? PASC_OK
               : PASC_ERR_HIP;
}

template <int K>
static int launch_k(const GridLoopArgs &a, int nwg, int npt, hipStream_t s) {
    return npt == 1 ? launch_kn<K, 1>(a, nwg, s)
                    : npt == 2 ? launch_kn<K, 2>(a, nwg, s) : launch_kn<K, 4>(a, nwg, s);
}

// PASC_ERR_HIP (without a message): the launch was refused, the caller runs the graph kernels
int LOOP_FN(int K, const GridLoopArgs &a, int nwg, int npt, hipStream_t s) {
    switch (K) {
        case 1: return launch_k<1>(a, nwg, npt, s);
        case 2: return launch_k<2>(a, nwg, npt, s);
        case 3: return launch_k<3>(a, nwg, npt, s);
        case 4: return launch_k<4>(a, nwg, npt, s);
        case 5: return launch_k<5>(a, nwg, npt, s);
        case 6: return launch_k<6>(a, nwg, npt, s);
        case 7: return launch_k<7>(a, nwg, npt, s);
        case 8: return launch_k<8>(a, nwg, npt, s);
    }
    return PASC_ERR_HIP;
}

}  // namespace pasc
