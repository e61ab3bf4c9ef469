// Instantiations of the persistent image loop for one storage type (PASS_S) and one number of rows
// per wave (LOOP_ROWS).
#include "img_loop.h"

#if !defined(PASS_S) || !defined(LOOP_ROWS)
#error "PASS_S (float or double) and LOOP_ROWS (image rows per wave) must be defined"
#endif

#define PASC_CAT3_(a, b, c) a##b##c
#define PASC_CAT3(a, b, c) PASC_CAT3_(a, b, c)
#define LOOP_FN PASC_CAT3(launch_img_loop_, PASS_S, PASC_CAT3(_, LOOP_ROWS, _))

namespace pasc {

template <int K, int NW>
static int launch_kn(const ImgLoopArgs &a, int nwg, hipStream_t s) {
    if constexpr (LOOP_ROWS <= img_loop_rows<PASS_S>(K)) {
        using L = ImgLoopShape<PASS_S, K, NW, LOOP_ROWS>;
        static_assert(L::LDS <= LOOP_LDS_BYTES && L::HN <= NW * WAVE, "one thread per halo node");
        const void *fn = reinterpret_cast<const void *>(img_loop<PASS_S, K, NW, LOOP_ROWS>);
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::LDS) != hipSuccess)
            return PASC_ERR_HIP;
        ImgLoopArgs args = a;
        void *params[] = {&args};
        return hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(NW * WAVE), params, (unsigned)L::LDS,
                                          s) == hipSuccess
                   ? PASC_OK
                   : PASC_ERR_HIP;
    }
    return PASC_ERR_HIP;
}

template <int K>
static int launch_k(const ImgLoopArgs &a, int nwg, int nw, hipStream_t s) {
#if LOOP_ROWS == 1
    if (nw == 4) return launch_kn<K, 4>(a, nwg, s);
#endif
    return nw == 8 ? launch_kn<K, 8>(a, nwg, s) : PASC_ERR_HIP;
}

// PASC_ERR_HIP (without a message): the launch was refused, the caller runs the image pass
int LOOP_FN(int K, const ImgLoopArgs &a, int nwg, int nw, hipStream_t s) {
    switch (K) {
        case 1: return launch_k<1>(a, nwg, nw, s);
        case 2: return launch_k<2>(a, nwg, nw, s);
        case 3: return launch_k<3>(a, nwg, nw, s);
        case 4: return launch_k<4>(a, nwg, nw, s);
        case 5: return launch_k<5>(a, nwg, nw, s);
        case 6: return launch_k<6>(a, nwg, nw, s);
        case 7: return launch_k<7>(a, nwg, nw, s);
        case 8: return launch_k<8>(a, nwg, nw, s);
    }
    return PASC_ERR_HIP;
}

}  // namespace pasc
