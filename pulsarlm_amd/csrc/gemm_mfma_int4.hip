// mfma_kernel for plain int4 calls.
#include "gemm_mfma.hpp"

namespace plm {

void launch_plain_int4(const mfma_args& a, bool bf16, bool uniform, int id, dim3 grid, hipStream_t s) {
    const int mode = (bf16 ? 4 : 0) + (uniform ? 2 : 0) + (a.scale_dtype == PLM_FP32 ? 1 : 0);
    switch (mode) {
        case 0: launch_shape<PLM_INT4, false, false, false, false>(a, id, grid, s); break;
        case 1: launch_shape<PLM_INT4, false, false, true, false>(a, id, grid, s); break;
        case 2: launch_shape<PLM_INT4, false, true, false, false>(a, id, grid, s); break;
        case 3: launch_shape<PLM_INT4, false, true, true, false>(a, id, grid, s); break;
        case 4: launch_shape<PLM_INT4, true, false, false, false>(a, id, grid, s); break;
        case 5: launch_shape<PLM_INT4, true, false, true, false>(a, id, grid, s); break;
        case 6: launch_shape<PLM_INT4, true, true, false, false>(a, id, grid, s); break;
        default: launch_shape<PLM_INT4, true, true, true, false>(a, id, grid, s); break;
    }
}

}  // namespace plm
