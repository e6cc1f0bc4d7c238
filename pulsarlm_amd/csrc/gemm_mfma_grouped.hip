// mfma_kernel for grouped (MoE) calls.
#include <algorithm>

#include "gemm_mfma.hpp"

namespace plm {

// Shapes of grouped calls.
namespace {
constexpr shape kGroupedShapes[7] = {kRows16, kRows64, kSmall, kLarge, kHuge, kRows32, kTall};
}

// Grouped: `tiles` holds max_tiles (expert, first row, rows) records built on the device;
// rows are in the grouped (sorted) order and `row_index` optionally gathers them from x.
// shape indexes kGroupedShapes (int4 experts only); 6 (256 x 256 tall) is for full blocks of rows.
namespace {
// PERSIST launches: about one workgroup per slot the kernel can hold resident (occupancy per CU
// times the CUs), a multiple of 8 so that every XCD gets the same number of workgroups, and
// never more than the items.
template <typename K>
unsigned persistent_grid(K kernel, int threads, unsigned items) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess || per_cu < 1)
        per_cu = 1;
    const unsigned slots = static_cast<unsigned>(per_cu * cu_count()) & ~7u;
    return std::max(8u, std::min(items, slots));
}

template <bool BF16, bool UNIFORM, bool WIDE, int I>
void launch_grouped_one(const mfma_args& a, dim3 grid, bool persist, hipStream_t s) {
    constexpr shape sh = kGroupedShapes[I];
    constexpr int threads = sh.wm * sh.wn * 64;
    if constexpr (I != 4) {  // the 256 x 256 two-row grid (unused by the MoE block) is never persistent
        if (persist) {
            auto* kernel = mfma_kernel<PLM_INT4, BF16, UNIFORM, WIDE, false, true, sh.wm, sh.wn, sh.mt, sh.ns, true, true>;
            grid.x = persistent_grid(kernel, threads, grid.x);
            kernel<<<grid, threads, 0, s>>>(a);
            return;
        }
    }
    mfma_kernel<PLM_INT4, BF16, UNIFORM, WIDE, false, true, sh.wm, sh.wn, sh.mt, sh.ns, true>
        <<<grid, threads, 0, s>>>(a);
}

template <bool BF16, bool UNIFORM, bool WIDE>
void launch_grouped_shape(const mfma_args& a, int shape, dim3 grid, bool persist, hipStream_t s) {
    switch (shape) {
        case 0: launch_grouped_one<BF16, UNIFORM, WIDE, 0>(a, grid, persist, s); break;
        case 1: launch_grouped_one<BF16, UNIFORM, WIDE, 1>(a, grid, persist, s); break;
        case 2: launch_grouped_one<BF16, UNIFORM, WIDE, 2>(a, grid, persist, s); break;
        case 3: launch_grouped_one<BF16, UNIFORM, WIDE, 3>(a, grid, persist, s); break;
        case 5: launch_grouped_one<BF16, UNIFORM, WIDE, 5>(a, grid, persist, s); break;
        case 6: launch_grouped_one<BF16, UNIFORM, WIDE, 6>(a, grid, persist, s); break;
        default: launch_grouped_one<BF16, UNIFORM, WIDE, 4>(a, grid, persist, s); break;
    }
}
}  // namespace

int grouped_block_rows(int shape) { return kGroupedShapes[std::min(std::max(shape, 0), 6)].bm(); }

// Row block for a grouped call, from the average rows per expert. At the Zipf-routed
// T = 256 block (16 rows per expert on average, the heaviest experts near 250) 32-row tiles
// measured 6 % faster than 16-row ones and 64-row ones 5 % slower: a weight tile is
// dequantized once per row block, and the dequant bounds these small GEMMs.
int grouped_rows_env() { return knobs().moe_rows; }  // PLM_MOE_ROWS=16/32/64 (tuning sweeps)
int grouped_shape_for(int64_t rows, int64_t n_experts) {
    const int64_t avg = ceil_div(rows, std::max<int64_t>(n_experts, 1));
    switch (grouped_rows_env()) {
        case 16: return 0;
        case 32: return 5;
        case 64: return 1;
        default: break;
    }
    if (avg <= 8) return 0;
    if (avg <= 24) return 5;
    if (avg <= 96) return 1;
    if (avg <= 192) return 2;
    return 3;
}

int launch_grouped(const char* op, plm_format f, const void* x, bool bf16, const void* w, const void* scale,
                   plm_dtype scale_dtype, int64_t rows, int64_t n, int64_t k, int64_t block_n, int64_t group_size,
                   void* y, const int32_t* tiles, int64_t max_tiles, const int32_t* tile_count,
                   const int32_t* row_index, int shape, hipStream_t s, bool swiglu) {
    PLM_CHECK_ARG(f == PLM_INT4, op, "grouped GEMMs take int4 experts");
    PLM_CHECK_ARG(k <= (int64_t{1} << 21) && rows * k * 2 < kOOB && n * k < (int64_t{1} << 40), op,
                  "problem too large");
    mfma_args a{};
    fill_common(a, x, w, scale, scale_dtype, rows, n, k, block_n, group_size, y);
    const struct shape sh = kGroupedShapes[std::min(std::max(shape, 0), 6)];
    a.splits = 1;
    a.tiles_per_split = a.ktiles;
    a.m_blocks = 1;
    a.n_blocks = static_cast<int>(ceil_div(a.strips, sh.bs()));
    if (swiglu) {  // [gate; up] with whole 16-column strips each: slices of bs / 2 strip pairs
        PLM_CHECK_ARG(n % (2 * kTileN) == 0 && sh.ns % 2 == 0, op, "fused activation needs 16 | intermediate");
        a.swiglu_strips = static_cast<int>(n / (2 * kTileN));
        a.n_blocks = static_cast<int>(ceil_div(a.swiglu_strips, sh.bs() / 2));
    }
    a.tiles = tiles;
    a.tile_count = tile_count;
    a.row_index = row_index;
    a.w_expert_bytes = ceil_div(n, kTileN) * ceil_div(k, kTileK) * tile_bytes(f);
    a.s_expert_bytes = static_cast<int64_t>(a.strips) * a.groups * a.scale_cols * dtype_size(scale_dtype);
    dim3 grid(static_cast<unsigned>(round_up(max_tiles * a.n_blocks, 8)), 1);  // whole XCD rounds
    const bool persist = knobs().moe_persist;  // A/B measurements: measured slower
    const bool uniform = group_size % kTileK == 0;
    const bool wide = scale_dtype == PLM_FP32;
    const int mode = (bf16 ? 4 : 0) + (uniform ? 2 : 0) + (wide ? 1 : 0);
    switch (mode) {
        case 0: launch_grouped_shape<false, false, false>(a, shape, grid, persist, s); break;
        case 1: launch_grouped_shape<false, false, true>(a, shape, grid, persist, s); break;
        case 2: launch_grouped_shape<false, true, false>(a, shape, grid, persist, s); break;
        case 3: launch_grouped_shape<false, true, true>(a, shape, grid, persist, s); break;
        case 4: launch_grouped_shape<true, false, false>(a, shape, grid, persist, s); break;
        case 5: launch_grouped_shape<true, false, true>(a, shape, grid, persist, s); break;
        case 6: launch_grouped_shape<true, true, false>(a, shape, grid, persist, s); break;
        default: launch_grouped_shape<true, true, true>(a, shape, grid, persist, s); break;
    }
    PLM_HIP_LAUNCH_CHECK(op);
    return PLM_OK;
}

}  // namespace plm
