// The fused quantized GEMV on k slices for at most four rows (qgemv_fused.hip has
// the rest of its forms and the launcher).
#include "common.h"
#include "kernels.h"
#include "qgemv_kernel.h"

namespace slhip {

hipError_t run_qgemv_sliced_few_rows(bool int4, int spg, dim3 grid, uint32_t threads, size_t lds, const float* a,
                                     const float* gamma, uint32_t mk, uint32_t k, const void* args, hipStream_t s) {
    const Args& p = *static_cast<const Args*>(args);
#define SL_QGEMV_SLICED(B, G) qgemv_fused<B, 1, G, true, 8, 16, true, kSmStream><<<grid, threads, lds, s>>>(a, gamma, mk, k, p)
    if (int4) {
        if (spg == 1) SL_QGEMV_SLICED(4, 1);
        else if (spg == 2) SL_QGEMV_SLICED(4, 2);
        else SL_QGEMV_SLICED(4, 0);
    } else {
        if (spg == 1) SL_QGEMV_SLICED(8, 1);
        else if (spg == 2) SL_QGEMV_SLICED(8, 2);
        else SL_QGEMV_SLICED(8, 0);
    }
#undef SL_QGEMV_SLICED
    return hipGetLastError();
}

// Loads this file's code object now: HIP loads one at the first use of
// any of its kernels, which otherwise lands inside the first submission
// that needs it (about 1-2 ms each, more for large objects).
hipError_t load_code_qgemv_sliced() {
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr,
                                reinterpret_cast<const void*>(&qgemv_fused<4, 1, 2, true, 8, 16, true, kSmStream>));
}

}  // namespace slhip
