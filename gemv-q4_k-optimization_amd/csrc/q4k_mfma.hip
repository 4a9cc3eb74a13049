// q4k_mfma.hip -- the matrix-core Q4_K GEMV kernels (q4k_mfma.h), in a
// translation unit of their own; q4k_gemv.hip picks their launch shapes.
#include <hip/hip_runtime.h>

#include "q4k_mfma.h"
#include "q4k_runtime.h"

namespace q4k {

template <int WAVES, bool SUMS>
static const void *mfma_kernel_nc(int nc) {
    switch (nc) {
        case 1: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<1, WAVES, SUMS>);
        case 2: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<2, WAVES, SUMS>);
        case 3: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<3, WAVES, SUMS>);
        case 4: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<4, WAVES, SUMS>);
        case 5: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<5, WAVES, SUMS>);
        case 6: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<6, WAVES, SUMS>);
        case 7: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<7, WAVES, SUMS>);
        case 8: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<8, WAVES, SUMS>);
        default: return nullptr;
    }
}

const void *q4k_mfma_kernel(int nc, int waves, bool sums) {
    if (waves > 8) return sums ? mfma_kernel_nc<16, true>(nc) : mfma_kernel_nc<16, false>(nc);
    return sums ? mfma_kernel_nc<8, true>(nc) : mfma_kernel_nc<8, false>(nc);
}

template <int NIF>
static const void *mfma_ga_kernel_nc(int nc) {
    switch (nc) {
        case 1: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<1, 8, false, true, NIF>);
        case 2: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<2, 8, false, true, NIF>);
        case 3: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<3, 8, false, true, NIF>);
        case 4: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<4, 8, false, true, NIF>);
        case 5: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<5, 8, false, true, NIF>);
        case 6: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<6, 8, false, true, NIF>);
        case 7: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<7, 8, false, true, NIF>);
        case 8: return reinterpret_cast<const void *>(&gemv_q4k_mfma_kernel<8, 8, false, true, NIF>);
        default: return nullptr;
    }
}

// GA: 8-wave workgroups, 2 or 4 items in flight per wave
const void *q4k_mfma_ga_kernel(int nc, int waves, int nif) {
    if (waves != 8) return nullptr;
    return nif == 4 ? mfma_ga_kernel_nc<4>(nc) : mfma_ga_kernel_nc<2>(nc);
}

}  // namespace q4k
