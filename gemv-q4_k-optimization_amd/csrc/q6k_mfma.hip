// q6k_mfma.hip -- the matrix-core Q6_K GEMV kernels (q6k_mfma.h), in a
// translation unit of their own; q6k_gemv.hip picks their launch shapes.
#include <hip/hip_runtime.h>

#include "q6k_mfma.h"
#include "q4k_runtime.h"

namespace q4k {

template <int WAVES>
static const void *q6_mfma_kernel_nc(int nc) {
    switch (nc) {
        case 1: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<1, WAVES>);
        case 2: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<2, WAVES>);
        case 3: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<3, WAVES>);
        case 4: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<4, WAVES>);
        case 5: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<5, WAVES>);
        case 6: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<6, WAVES>);
        case 7: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<7, WAVES>);
        case 8: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<8, WAVES>);
        default: return nullptr;
    }
}

const void *q6k_mfma_kernel(int nc, int waves) {
    return waves > 8 ? q6_mfma_kernel_nc<16>(nc) : q6_mfma_kernel_nc<8>(nc);
}

// GA: 8-wave workgroups
const void *q6k_mfma_ga_kernel(int nc, int waves) {
    if (waves != 8) return nullptr;
    switch (nc) {
        case 1: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<1, 8, false, true>);
        case 2: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<2, 8, false, true>);
        case 3: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<3, 8, false, true>);
        case 4: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<4, 8, false, true>);
        case 5: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<5, 8, false, true>);
        case 6: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<6, 8, false, true>);
        case 7: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<7, 8, false, true>);
        case 8: return reinterpret_cast<const void *>(&gemv_q6k_mfma_kernel<8, 8, false, true>);
        default: return nullptr;
    }
}

}  // namespace q4k
