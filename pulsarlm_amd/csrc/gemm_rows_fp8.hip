// rows_kernel for fp8 (e4m3) weights with bf16 / fp16 activations: fp32 scales, per column or per
// 16-column strip, groups a multiple of 128 (the checkpoint forms).
#include "gemm_rows.hpp"

namespace plm {

namespace {

template <bool BF16, int SCM, int RB>
bool launch_sg(const rows_args& a, int sg, dim3 grid, size_t lds, hipStream_t s) {
    switch (sg) {
        case 1: rows_kernel<PLM_FP8, BF16, SCM, false, RB, 1><<<grid, kRowsWaves * 64, lds, s>>>(a); return true;
        case 2: rows_kernel<PLM_FP8, BF16, SCM, false, RB, 2><<<grid, kRowsWaves * 64, lds, s>>>(a); return true;
        case 3: rows_kernel<PLM_FP8, BF16, SCM, false, RB, 3><<<grid, kRowsWaves * 64, lds, s>>>(a); return true;
        case 4: rows_kernel<PLM_FP8, BF16, SCM, false, RB, 4><<<grid, kRowsWaves * 64, lds, s>>>(a); return true;
        default: return false;
    }
}

template <bool BF16, int SCM>
bool launch_rb(const rows_args& a, int rb, int sg, dim3 grid, size_t lds, hipStream_t s) {
    switch (rb) {
        case 1: return launch_sg<BF16, SCM, 1>(a, sg, grid, lds, s);
        case 2: return launch_sg<BF16, SCM, 2>(a, sg, grid, lds, s);
        case 3: return launch_sg<BF16, SCM, 3>(a, sg, grid, lds, s);
        case 4: return launch_sg<BF16, SCM, 4>(a, sg, grid, lds, s);
        default: return false;
    }
}

}  // namespace

template <>
bool launch_rows_shape<PLM_FP8>(const rows_args& a, bool bf16, int scm, bool sub, int rb, int sg, dim3 grid, size_t lds,
                                hipStream_t s) {
    if (sub || (scm != 1 && scm != 2)) return false;
    if (bf16) return scm == 1 ? launch_rb<true, 1>(a, rb, sg, grid, lds, s) : launch_rb<true, 2>(a, rb, sg, grid, lds, s);
    return scm == 1 ? launch_rb<false, 1>(a, rb, sg, grid, lds, s) : launch_rb<false, 2>(a, rb, sg, grid, lds, s);
}

}  // namespace plm
