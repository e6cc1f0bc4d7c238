// mfma_kernel for W8A8 calls.
#include "gemm_mfma.hpp"

namespace plm {

void launch_plain_a8(const mfma_args& a, bool bf16, int id, dim3 grid, hipStream_t s) {
    const bool wide = a.scale_dtype == PLM_FP32;
    if (bf16 && wide) launch_shape<PLM_FP8, true, true, true, true>(a, id, grid, s);
    else if (bf16) launch_shape<PLM_FP8, true, true, false, true>(a, id, grid, s);
    else if (wide) launch_shape<PLM_FP8, false, true, true, true>(a, id, grid, s);
    else launch_shape<PLM_FP8, false, true, false, true>(a, id, grid, s);
}

}  // namespace plm
