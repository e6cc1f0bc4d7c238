// MFMA dequant-GEMM for larger row counts (prefill), its W8A8 form and its grouped (MoE) form:
// y[M, N] = x[M, K] @ dequant(W)^T.
//
// Counterpart of the reference's marlin_kernel at tile_m = 64 (pulsarlm-core/src/kernels/
// marlin.cu:251-389; dispatch :577-596) with its split-K combine
// (pulsarlm-core/inc/pulsarlm/kernels/dequant_gemm_common.cuh:99-133), and, in grouped
// mode, of one at::_grouped_mm of routed_experts (pulsarlm-core/src/engine/model/
// paged_forward.cpp:124-125).
//
// gfx950 design:
// * Workgroup tile (WM*MT*16) x (WN*NS*16) over 128-wide K steps; WM x WN wavefronts,
//   each owning MT x NS tiles of v_mfma_f32_16x16x32 (bf16/fp16). Most shapes have one row
//   of wavefronts, so every strip is dequantized by one wavefront only and each dequantized
//   weight feeds MT MFMAs (a second row of wavefronts would dequantize each strip twice).
// * The x tile and the packed weight tiles (1 KiB int4 / 2 KiB fp8 per 16-column strip,
//   copied verbatim from the plm layout) go from HBM straight into LDS with buffer loads to
//   LDS (no register staging), double-buffered: the next K step's loads land in one stage
//   while the current step's MFMAs read the other, with one barrier per K step. x rows are
//   XOR-swizzled in LDS so that fragment reads are free of bank conflicts; rows past M and
//   columns past K read as zeros through the buffer range instead of branches.
// * Weights are dequantized in registers to round(q * round(s)), bit-identical to the
//   reference's fragment values (shared dq_int4 / dq_fp8).
// * A8 (W8A8): x is e4m3 (quantized per row beforehand) and every 128-wide K tile is one
//   v_mfma_scale_f32_16x16x128_f8f6f4 per output tile on the raw weight bytes; the tile's
//   partial is scaled by the weight block scale and, at the end, by the row scale.
// * Grouped: each work tile is (expert, block of that expert's rows); rows may be gathered
//   through a row index (the tokens routed to the expert) and the expert's weights and
//   scales are found at a fixed stride.
// * Split-K across workgroups when the output has too few tiles to fill the GPU, reduced
//   deterministically by the last workgroup to arrive.
// * Grouped gate_up of the MoE block may fuse the activation: the workgroup's local strips
//   2p and 2p + 1 are the gate and up strips of one 16-column slice, so every wavefront
//   holds both halves of its outputs and the epilogue writes act = round(round(silu(g)) *
//   u) (the unfused silu_mul's expression) instead of the [rows, 2I] gate_up product.
#pragma once

#include <type_traits>

#include "plm_common.hpp"

namespace plm {

struct mfma_args {
    const uint16_t* x;
    const uint8_t* w;
    const void* scale;
    uint16_t* y;
    float* partial;
    uint32_t* counters;
    int scale_dtype, scale_cols;
    int m, n, k;
    int ktiles, strips, groups, group_size;
    float group_inv;  // 16 / group_size
    int splits, tiles_per_split;
    int m_blocks, n_blocks;
    int tile_base;  // plain calls: this launch's work tiles start at tile_base
    int xcd_rows;   // plain calls: row blocks of an XCD's patch of work tiles (0: tiles in id order)
    // A8
    const uint8_t* xq;      // e4m3 [M][ktiles][128], lane-permuted within each tile
    const float* x_scale;   // [M]
    // Grouped
    const int32_t* tiles;      // [max_tiles][3]: expert, first row, rows (rows == 0: idle)
    const int32_t* tile_count;  // the number of real tiles (a prefix of `tiles`)
    const int32_t* row_index;  // gather: A row r is x[row_index[r]] (null: x[r])
    int64_t w_expert_bytes;
    int64_t s_expert_bytes;
    // Grouped gate_up with the activation fused (0: off): the weight is [gate; up] with
    // swiglu_strips 16-column strips each; a workgroup takes gate strip p and up strip
    // swiglu_strips + p side by side and writes round(round(silu(g)) * u) into y [rows, 16 *
    // swiglu_strips] instead of the [rows, 2I] product.
    int swiglu_strips;
};

namespace {

// K splits whose partial sums the last workgroup of a tile loads at a time.
constexpr int split_batch(int mt, int ns) { return mt * ns <= 4 ? 8 : (mt * ns <= 8 ? 4 : (mt * ns <= 16 ? 2 : 1)); }

template <bool A8> struct a_traits {
    static constexpr int row_bytes = A8 ? kTileK : kTileK * 2;  // one A row of one K tile
    static constexpr int slots = row_bytes / 16;                 // its 16-byte slots
};

// VO: the 16-byte epilogue (see its comment) is compiled in; the host selects it per launch.
template <plm_format F, bool BF16, bool UNIFORM, bool WIDE, bool A8, bool GROUPED, int WM, int WN, int MT, int NS,
          bool VO = false, bool PERSIST = false>
__global__ void __launch_bounds__(WM * WN * 64) mfma_kernel(mfma_args a) {
    constexpr int NW = WM * WN;  // wavefronts
    constexpr int NT = NW * 64;
    constexpr int TB = fmt_traits<F>::tile_bytes;
    constexpr int BM = WM * MT * 16;
    constexpr int BS = WN * NS;  // strips per workgroup
    constexpr int ARB = a_traits<A8>::row_bytes;
    constexpr int SLOTS = a_traits<A8>::slots;
    constexpr int RPC = 1024 / ARB;  // A rows per 1 KiB chunk
    constexpr int A_STAGE = BM * ARB;
    // fp8 W8A16 with one row of wavefronts: no two wavefronts share a weight strip, so each
    // loads its own strips' tiles for the next K step into registers and LDS holds only x
    // (the 2 KiB fp8 tiles of 16 strips would not fit beside two 64 KiB x stages). int4's
    // 1 KiB tiles fit; loading them the same way measured 8 % slower at M = 4096.
    constexpr bool BREG = F == PLM_FP8 && !A8 && !GROUPED && WM == 1;
    constexpr int B_STAGE = BREG ? 0 : BS * TB;
    constexpr int STAGE = A_STAGE + B_STAGE;
    constexpr int A_CHUNKS = A_STAGE / 1024, B_CHUNKS = B_STAGE / 1024;
    constexpr int A_PW = (A_CHUNKS + NW - 1) / NW;  // 1 KiB chunks each wavefront loads per K step
    constexpr int B_PW = (B_CHUNKS + NW - 1) / NW;
    static_assert(A_STAGE % 1024 == 0 && B_STAGE % 1024 == 0, "stages are whole 1 KiB chunks");
    constexpr int ST = UNIFORM ? 1 : 4;  // scale values per strip per K step
    constexpr int ES = WIDE ? 4 : 2;     // scale element bytes
    // Software-pipelined x fragments (see the K loop), for the one-row tall shapes.
    constexpr bool PIPE_A = UNIFORM && !A8 && WM == 1 && MT >= 8;
    // The same for W8A8 on the shapes that run one workgroup to a CU (K 4096, N 6144: M = 2048 60.1 ->
    // 58.3 us, M = 4096 110.3 -> 106.4; K 17408, N 5120, M = 2048 209 -> 205). With two or three
    // workgroups others fill the waits, and a fixed order costs 2-3 % (K 8192, N 2048, M = 3300).
    constexpr bool PIPE_A8 = A8 && WM * WN == 8 && NS > 1;
    // Fragments kept a slice ahead: all MT, or 12 for fp8, whose weight tiles already hold
    // two K steps of registers (16 would spill).
    // PERSIST keeps 8 fewer: the item loop needs the registers (the tall tile spills otherwise).
    constexpr int PD = F == PLM_FP8 ? MT - 4 : (PERSIST ? MT - 8 : MT);

    // Two stages of [A tile | weight tiles]. Stage s holds K step kt_begin + s (mod 2); the
    // loads of step kt + 1 go straight from HBM into the other stage while step kt computes.
    // The split-K arrival flag reuses the first word once the K loop is over (arrive_last
    // synchronizes the workgroup before writing it).
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * STAGE];
    uint32_t& last_flag = *reinterpret_cast<uint32_t*>(lds);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int col16 = lane & 15, kq = lane >> 4;
    const int split = blockIdx.y;
    const bool swiglu = GROUPED && a.swiglu_strips > 0;
    const int kt_begin = split * a.tiles_per_split;
    const int kt_end = min(kt_begin + a.tiles_per_split, a.ktiles);
    const int a_stride = A8 ? a.ktiles * kTileK : a.k * 2;
    const int strip_bytes = a.ktiles * TB;
    const bool bf16_scale = a.scale_dtype == PLM_BF16;
    const int s_row = a.groups * a.scale_cols * ES;  // scale bytes per strip
    const int s_lane = a.scale_cols == 1 ? 0 : col16 * ES;
    const int lrow = lane / SLOTS, lslot = lane % SLOTS;

    // Work items: plain calls take work tile blockIdx.x + tile_base (row block fastest);
    // grouped calls take (expert tile, column block) items. Workgroups are dealt to the 8
    // XCDs round-robin by id, so a grouped call gives out its real items in 8 contiguous runs,
    // one per XCD: the column blocks of a row tile (the same x rows) and the consecutive
    // tiles of an expert (the same weights) run on one XCD and share its L2; ids past the
    // real items exit. PERSIST (grouped only; an A/B option, measured slower than one item
    // per workgroup): the grid holds about one workgroup per slot the CUs keep resident, each
    // workgroup walks its XCD's run gridDim.x / 8 items apart and loads the next item's first
    // K step into the free LDS stage during the current item's epilogue.
    static_assert(!PERSIST || (GROUPED && !A8), "persistent launches are grouped ones");
    int items = 0, per_xcd = 0;
    if constexpr (GROUPED) {
        items = uniform(*a.tile_count) * a.n_blocks;
        per_xcd = (items + 7) >> 3;
    }
    auto item_at = [&](int pos) -> int {  // this workgroup's pos-th item, -1 past its last
        if constexpr (GROUPED) {
            const int idx = (blockIdx.x >> 3) + pos * (gridDim.x >> 3);
            if (idx >= per_xcd) return -1;
            const int it = (blockIdx.x & 7) * per_xcd + idx;
            return it < items ? it : -1;
        } else {
            return blockIdx.x + a.tile_base;
        }
    };

    // Everything that depends on the item: output tile, and the buffers and per-lane offsets
    // of its A rows, weight strips and scales.
    struct item_ctx {
        int nb, row0, rows;
        __amdgpu_buffer_rsrc_t a_rsrc, b_rsrc, s_rsrc;
        int a_gather[GROUPED ? A_PW : 1];  // grouped: the gathered rows' offsets
        int b_off[B_PW > 0 ? B_PW : 1];
        int s_strip[NS];  // byte offset of strip j's scales in s_rsrc
    };
    // SwiGLU (grouped): local strip s is gate strip (s even) or up strip (s odd) of slice
    // nb * BS / 2 + s / 2; otherwise strip strip0 + s.
    auto wstrip = [&](int nb, int s_local) -> int {
        if (swiglu) {
            const int slice = nb * (BS / 2) + (s_local >> 1);
            return slice < a.swiglu_strips ? slice + ((s_local & 1) ? a.swiglu_strips : 0) : -1;
        }
        return nb * BS + s_local < a.strips ? nb * BS + s_local : -1;
    };
    auto locate = [&](int item, item_ctx& c) -> bool {  // false: an idle grouped tile
        int expert = 0;
        if constexpr (GROUPED) {
            const int tile = item / a.n_blocks;
            c.nb = item % a.n_blocks;
            expert = a.tiles[3 * tile];
            c.row0 = a.tiles[3 * tile + 1];
            c.rows = a.tiles[3 * tile + 2];
            if (c.rows <= 0) return false;  // uniform across the workgroup
        } else {
            int mb;
            if (a.xcd_rows > 0) {
                // Workgroups go round the 8 XCDs by id: each takes one run of the work tiles, which
                // are ordered in bands of xcd_rows row blocks, row block fastest.
                const int tiles = a.m_blocks * a.n_blocks, x = item & 7;
                const int lin = x * (tiles >> 3) + min(x, tiles & 7) + (item >> 3);
                const int band = lin / (a.xcd_rows * a.n_blocks), first = band * a.xcd_rows;
                const int rows = min(a.xcd_rows, a.m_blocks - first), in = lin - first * a.n_blocks;
                c.nb = in / rows;
                mb = first + in % rows;
            } else {
                c.nb = item / a.m_blocks;
                mb = item % a.m_blocks;
            }
            c.row0 = mb * BM;
            c.rows = min(BM, a.m - c.row0);
        }
        const int strip0 = c.nb * BS;
        // PERSIST: lane-derived offsets come from an opaque copy of the lane id, so that the
        // compiler recomputes them per item instead of hoisting them out of the item loop and
        // keeping them live across the K loop (the tall tile has no registers to spare).
        int llane = lane;
        if constexpr (PERSIST) asm volatile("" : "+v"(llane));
        const int lrow_l = llane / SLOTS;
        const uint8_t* wbase = a.w + (GROUPED ? expert * a.w_expert_bytes : 0);
        const uint8_t* sbase = static_cast<const uint8_t*>(a.scale) + (GROUPED ? expert * a.s_expert_bytes : 0);
        // A source: row-major rows of ARB bytes per K tile. Plain calls address rows from row0
        // and bound the buffer at `rows` rows; grouped calls gather rows through row_index
        // (the host checks every offset stays below kOOB) and keep the offsets in registers.
        if constexpr (GROUPED) {
            c.a_rsrc = make_rsrc(a.x, static_cast<uint32_t>(kOOB));
#pragma unroll
            for (int i = 0; i < A_PW; ++i) {
                const int r = (wave * A_PW + i) * RPC + lrow_l;
                int src = -1;
                if (r < c.rows) src = a.row_index != nullptr ? a.row_index[c.row0 + r] : c.row0 + r;
                c.a_gather[i] = src < 0 ? kOOB : src * a_stride;
            }
        } else {
            const uint8_t* base = A8 ? a.xq : reinterpret_cast<const uint8_t*>(a.x);
            c.a_rsrc = make_rsrc(base + static_cast<int64_t>(c.row0) * a_stride, static_cast<uint32_t>(c.rows * a_stride));
        }
        // Weights: this workgroup's strips are contiguous, ktiles * TB bytes each (with SwiGLU,
        // two runs of them, addressed from the expert's first strip).
        c.b_rsrc = swiglu ? make_rsrc(wbase, static_cast<uint32_t>(a.strips * strip_bytes))
                          : make_rsrc(wbase + static_cast<int64_t>(strip0) * strip_bytes,
                                      static_cast<uint32_t>(min(BS, a.strips - strip0) * strip_bytes));
#pragma unroll
        for (int i = 0; i < B_PW; ++i) {
            const int ch = wave * B_PW + i;
            const int sl = ch / (TB / 1024), in_strip = (ch % (TB / 1024)) * 1024 + llane * 16;
            if (swiglu) {
                const int ws = wstrip(c.nb, sl);
                c.b_off[i] = ws >= 0 ? ws * strip_bytes + in_strip : kOOB;
            } else {
                c.b_off[i] = sl * strip_bytes + in_strip;
            }
        }
        // Scales of this workgroup's strips ([strip][group][scale_cols], ES bytes each); strips
        // past N read as zero.
        c.s_rsrc = swiglu ? make_rsrc(sbase, static_cast<uint32_t>(a.strips * s_row))
                          : make_rsrc(sbase + static_cast<int64_t>(strip0) * s_row,
                                      static_cast<uint32_t>(min(BS, a.strips - strip0) * s_row));
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            if (swiglu) {
                const int ws = wstrip(c.nb, wn * NS + j);
                c.s_strip[j] = ws >= 0 ? ws * s_row : kOOB;
            } else {
                c.s_strip[j] = (wn * NS + j) * s_row;
            }
        }
        return true;
    };

    // Chunk c of the A tile is rows c*RPC .. c*RPC+RPC-1; lane L of its load writes slot L % SLOTS
    // of row c*RPC + L / SLOTS, which holds the row's 16-byte column (slot ^ row % SLOTS): the XOR
    // swizzle puts the 16 rows of one MFMA fragment read in 16 different bank groups.
    // Plain calls recompute the offsets per load (rows past `rows` fall outside the buffer).
    auto a_offset = [&](const item_ctx& c, int i, int kt) -> int {
        const int r = (wave * A_PW + i) * RPC + lrow;
        const int col = lslot ^ (r % SLOTS);
        const int row_off = GROUPED ? c.a_gather[GROUPED ? i : 0] : r * a_stride;
        if constexpr (!UNIFORM) {
            if (kt * kTileK + col * 8 >= a.k) return kOOB;  // K tail (bf16 x only)
        }
        return row_off + col * 16;
    };
    auto load_breg = [&](const item_ctx& c, u32x4_t (&dst)[NS][TB / 1024], int kt) {
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
            for (int h = 0; h < TB / 1024; ++h)
                dst[j][h] = buffer_load16(c.b_rsrc, (wn * NS + j) * strip_bytes + h * 1024 + lane * 16, kt * TB);
    };
    auto issue = [&](const item_ctx& c, int kt, int stage) {
        uint8_t* sa = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < A_PW; ++i)
            if (A_CHUNKS % NW == 0 || wave * A_PW + i < A_CHUNKS)  // wave-uniform
                buffer_load_lds16(c.a_rsrc, sa + (wave * A_PW + i) * 1024, a_offset(c, i, kt), kt * ARB);
#pragma unroll
        for (int i = 0; i < B_PW; ++i)
            if (B_CHUNKS % NW == 0 || wave * B_PW + i < B_CHUNKS)  // wave-uniform
                buffer_load_lds16(c.b_rsrc, sa + A_STAGE + (wave * B_PW + i) * 1024, c.b_off[i], kt * TB);
    };
    // Scales are loaded as raw bits one K step ahead and converted when used, so that no wait
    // on them stalls the tile loads in flight.
    auto scale_bits = [&](const item_ctx& c, int j, int kt, int t) -> uint32_t {
        int voff = s_lane + c.s_strip[j], soff = 0;
        if constexpr (UNIFORM) soff = uniform(kt * kTileK / a.group_size) * a.scale_cols * ES;
        else {
            // K / group_size from the fp32 reciprocal: exact below K = 2^25, since (K / 16 + 1/2) / (g / 16) is
            // at least 1 / (2 g / 16) from an integer. An integer division takes some 20
            // instructions, four times a strip and step (the MoE block with 64-wide groups, T = 1148: 1.075x).
            const float k16 = static_cast<float>((kt * kTileK + 32 * t + 8 * kq) >> 4);
            const int g = static_cast<int>(__builtin_fmaf(k16, a.group_inv, 0.5f * a.group_inv));
            voff += g * a.scale_cols * ES;
        }
        if constexpr (WIDE) return buffer_load_u32(c.s_rsrc, voff, soff);
        else return buffer_load_u16(c.s_rsrc, voff, soff);
    };

    // Epilogue: lane holds column col16 of strip (strip0 + wn*NS + j), rows 4*kq + r of m tile i.
    auto epilogue = [&](const item_ctx& c, f32x4_t (&acc)[MT][NS], int last_stage) {
        const int strip0 = c.nb * BS;
        int ekq = kq, ecol = col16, elane = lane;
        if constexpr (PERSIST) asm volatile("" : "+v"(ekq), "+v"(ecol), "+v"(elane));
        if constexpr (GROUPED && NS % 2 == 0) {
            if (swiglu) {  // gate strip j, up strip j + 1 of slice nb * BS / 2 + (wn * NS + j) / 2
                const int inter = a.swiglu_strips * kTileN;
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NS; j += 2) {
                        const int col = (c.nb * (BS / 2) + (wn * NS + j) / 2) * kTileN + ecol;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int lr = wm * MT * 16 + i * 16 + 4 * ekq + r;
                            if (lr < c.rows && col < inter)
                                a.y[static_cast<int64_t>(c.row0 + lr) * inter + col] = static_cast<uint16_t>(
                                    to_bits16<BF16>(silu_times<BF16>(round_to<BF16>(acc[i][j][r]),
                                                                     round_to<BF16>(acc[i][j + 1][r]))));
                        }
                    }
                return;
            }
        }
        // With 16-byte aligned output rows, each m tile goes through the wavefront's own LDS area
        // (16 rows of 16 * NS columns; the row pitch is padded by 16 bytes so the four row groups
        // of one write land in different banks) and leaves as one 16-byte store per 8 columns of
        // a row, instead of a 2-byte store per element. Separate instantiations (VO) for the
        // launches that take it: compiled into the split-K kernels too, it changed their register
        // allocation and made down at M = 1024 10 % slower. PERSIST stages in the stage the last
        // K step read (the other one holds the next item's first loads).
        if (VO && a.splits == 1 && (a.n & 7) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0) {
            constexpr int EROW = 32 * NS + 16;
            static_assert(!VO || 1024 + NW * 16 * EROW <= (PERSIST ? STAGE : 2 * STAGE), "epilogue staging fits");
            __syncthreads();  // every wavefront is past the K loop's last reads of the stages
            // Past the split-K arrival flag.
            uint8_t* ew = lds + (PERSIST ? last_stage * STAGE : 0) + 1024 + wave * 16 * EROW;
            const int col0 = (strip0 + wn * NS) * kTileN;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
#pragma unroll
                for (int j = 0; j < NS; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        *reinterpret_cast<uint16_t*>(ew + (4 * ekq + r) * EROW + (16 * j + ecol) * 2) =
                            static_cast<uint16_t>(to_bits16<BF16>(acc[i][j][r]));
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int c0 = 0; c0 < 32 * NS; c0 += 64) {  // 16 rows x 2 * NS chunks of 8 columns
                    const int ch16 = c0 + elane;
                    if (ch16 < 32 * NS) {
                        const int row = ch16 / (2 * NS), ch = ch16 % (2 * NS);
                        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ew + row * EROW + ch * 16);
                        const int lr = wm * MT * 16 + i * 16 + row;
                        const int col = col0 + ch * 8;
                        if (lr < c.rows && col < a.n)
                            *reinterpret_cast<u32x4_t*>(a.y + static_cast<int64_t>(c.row0 + lr) * a.n + col) = v;
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                const int col = (strip0 + wn * NS + j) * kTileN + ecol;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int lr = wm * MT * 16 + i * 16 + 4 * ekq + r;
                    if (lr < c.rows && col < a.n)
                        a.y[static_cast<int64_t>(c.row0 + lr) * a.n + col] =
                            static_cast<uint16_t>(to_bits16<BF16>(acc[i][j][r]));
                }
            }
    };

    int pos = 0;
    int item = item_at(0);
    if (item < 0) return;
    item_ctx cur;
    while (!locate(item, cur)) {
        if (!PERSIST) return;
        item = item_at(++pos);
        if (item < 0) return;
    }
    int stage0 = 0;      // the stage of this item's first K step
    bool loaded = false;  // its first K step is already in flight (PERSIST)
    for (;;) {
        f32x4_t acc[MT][NS];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NS; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

        uint32_t sc[NS][ST];
        u32x4_t wreg[NS][TB / 1024], wnext[NS][TB / 1024];  // BREG: this and the next step's tiles
        if (kt_begin < kt_end) {
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
                for (int t = 0; t < ST; ++t) sc[j][t] = scale_bits(cur, j, kt_begin, t);
            if (!loaded) issue(cur, kt_begin, stage0);
            if constexpr (BREG) load_breg(cur, wreg, kt_begin);
        }

        for (int kt = kt_begin; kt < kt_end; ++kt) {
            const int stage = stage0 ^ ((kt - kt_begin) & 1);
            // This step's tiles have landed (they are the only loads in flight) and every
            // wavefront is done with the other stage, which the next loads overwrite.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            uint32_t scn[NS][ST];
            const bool more = kt + 1 < kt_end;
            if (more) {
#pragma unroll
                for (int j = 0; j < NS; ++j)
#pragma unroll
                    for (int t = 0; t < ST; ++t) scn[j][t] = scale_bits(cur, j, kt + 1, t);
                issue(cur, kt + 1, stage ^ 1);
                if constexpr (BREG) load_breg(cur, wnext, kt + 1);
            }

            const uint8_t* sa = lds + stage * STAGE;
            const uint8_t* sb = sa + A_STAGE;
            u32x4_t wv[NS][TB / 1024];
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
                for (int h = 0; h < TB / 1024; ++h)
                    wv[j][h] = BREG ? wreg[j][h]
                                    : *reinterpret_cast<const u32x4_t*>(sb + (wn * NS + j) * TB + h * 1024 + lane * 16);

            auto frag_a8 = [&](int i) {
                const uint8_t* ra = sa + (wm * MT * 16 + i * 16 + col16) * ARB;
                const u32x4_t a0 = *reinterpret_cast<const u32x4_t*>(ra + (((2 * kq) ^ (col16 & 7)) * 16));
                const u32x4_t a1 = *reinterpret_cast<const u32x4_t*>(ra + (((2 * kq + 1) ^ (col16 & 7)) * 16));
                return __builtin_bit_cast(i32x8_t, u32x8_cat(a0, a1));
            };
            if constexpr (PIPE_A8) {
                // AD x fragments are read ahead of their MFMAs, and a product joins its accumulators
                // (times the block's scale) only after the next row of MFMAs is under way: left to
                // itself the compiler reads one fragment ahead and waits for it eight times a step.
                constexpr int AD = MT > 8 ? 2 : 4;
                i32x8_t af[AD];
#pragma unroll
                for (int i = 0; i < AD; ++i) af[i] = frag_a8(i);
                f32x4_t part[2][NS];
#pragma unroll
                for (int i = 0; i <= MT; ++i) {
#pragma unroll
                    for (int j = 0; j < NS; ++j) {
                        if (i < MT)
                            part[i & 1][j] = mfma16x16x128_fp8(
                                af[i % AD], __builtin_bit_cast(i32x8_t, u32x8_cat(wv[j][0], wv[j][TB / 1024 - 1])),
                                f32x4_t{0.f, 0.f, 0.f, 0.f});
                        if (i > 0)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[i - 1][j][r] = __builtin_fmaf(scale_from_bits<WIDE>(sc[j][0], bf16_scale),
                                                                  part[(i - 1) & 1][j][r], acc[i - 1][j][r]);
                        if (j == NS - 1 && i + AD < MT) af[i % AD] = frag_a8(i + AD);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            } else if constexpr (A8) {
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const i32x8_t av = frag_a8(i);
#pragma unroll
                    for (int j = 0; j < NS; ++j) {
                        const i32x8_t bv = __builtin_bit_cast(i32x8_t, u32x8_cat(wv[j][0], wv[j][TB / 1024 - 1]));
                        const f32x4_t part = mfma16x16x128_fp8(av, bv, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(scale_from_bits<WIDE>(sc[j][0], bf16_scale), part[r], acc[i][j][r]);
                    }
                }
            } else if constexpr (PIPE_A) {
                // The MT x fragments of a K slice are held in registers and each is re-read for
                // the next slice right after its MFMAs, so a fragment read has a whole slice of
                // MFMAs (MT * NS) to land instead of the next two.
                auto frag = [&](int i, int t) {
                    const uint8_t* ra = sa + (wm * MT * 16 + i * 16 + col16) * ARB;
                    return *reinterpret_cast<const u32x4_t*>(ra + (((4 * t + kq) ^ col16) * 16));
                };
                u32x4_t af[PD];
#pragma unroll
                for (int i = 0; i < PD; ++i) af[i] = frag(i, 0);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    u32x4_t b[NS];
#pragma unroll
                    for (int j = 0; j < NS; ++j) {
                        const float raw = scale_from_bits<WIDE>(sc[j][UNIFORM ? 0 : t], bf16_scale);
                        if constexpr (F == PLM_INT4) {
                            b[j] = dq_int4<BF16>(wv[j][0][t], make_int4_scale<BF16>(raw));
                        } else {
                            b[j] = dq_fp8<BF16>(wv[j][t >> 1][(t & 1) * 2], wv[j][t >> 1][(t & 1) * 2 + 1],
                                                round_to<BF16>(raw));
                        }
                    }
#pragma unroll
                    for (int i = 0; i < PD; ++i) {
#pragma unroll
                        for (int j = 0; j < NS; ++j) acc[i][j] = mfma16x16x32<BF16>(af[i], b[j], acc[i][j]);
                        if (t < 3) af[i] = frag(i, t + 1);
                        __builtin_amdgcn_sched_barrier(0);  // keep the read here, a slice ahead
                    }
#pragma unroll
                    for (int i = PD; i < MT; ++i) {
                        const u32x4_t a1 = frag(i, t);
#pragma unroll
                        for (int j = 0; j < NS; ++j) acc[i][j] = mfma16x16x32<BF16>(a1, b[j], acc[i][j]);
                    }
                }
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    // Dequantize this 32-wide K slice of every strip once, then stream the x
                    // fragments past it: each weight fragment feeds MT MFMAs.
                    u32x4_t b[NS];
#pragma unroll
                    for (int j = 0; j < NS; ++j) {
                        const float raw = scale_from_bits<WIDE>(sc[j][UNIFORM ? 0 : t], bf16_scale);
                        if constexpr (F == PLM_INT4) {
                            b[j] = dq_int4<BF16>(wv[j][0][t], make_int4_scale<BF16>(raw));
                        } else {
                            b[j] = dq_fp8<BF16>(wv[j][t >> 1][(t & 1) * 2], wv[j][t >> 1][(t & 1) * 2 + 1],
                                                round_to<BF16>(raw));
                        }
                    }
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const uint8_t* ra = sa + (wm * MT * 16 + i * 16 + col16) * ARB;
                        const u32x4_t af = *reinterpret_cast<const u32x4_t*>(ra + (((4 * t + kq) ^ col16) * 16));
#pragma unroll
                        for (int j = 0; j < NS; ++j) acc[i][j] = mfma16x16x32<BF16>(af, b[j], acc[i][j]);
                    }
                }
            }
            if (more) {
#pragma unroll
                for (int j = 0; j < NS; ++j)
#pragma unroll
                    for (int t = 0; t < ST; ++t) sc[j][t] = scn[j][t];
                if constexpr (BREG) {
#pragma unroll
                    for (int j = 0; j < NS; ++j)
#pragma unroll
                        for (int h = 0; h < TB / 1024; ++h) wreg[j][h] = wnext[j][h];
                }
            }
        }
        // The stage the last K step read; the other one is free.
        const int last_stage = stage0 ^ ((kt_end - 1 - kt_begin) & 1);

        // PERSIST: the next item's first K step goes into the free stage now, so that its loads
        // are in flight during this item's epilogue (which stages through last_stage only).
        int next = -1;
        item_ctx nxt;
        if constexpr (PERSIST) {
            for (;;) {
                next = item_at(++pos);
                if (next < 0 || locate(next, nxt)) break;
            }
            if (next >= 0) issue(nxt, kt_begin, last_stage ^ 1);
        }

        if constexpr (A8) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = cur.row0 + wm * MT * 16 + i * 16 + 4 * kq + r;
                    const float sx = a.x_scale[min(row, a.m - 1)];
#pragma unroll
                    for (int j = 0; j < NS; ++j) acc[i][j][r] *= sx;
                }
        }

        // Split K (never PERSIST): every workgroup stores its accumulators in lane order (16
        // bytes per lane per MFMA tile, so each store instruction is one contiguous 1 KiB) into
        // its own slot of the work tile's partial area; the last workgroup to arrive reloads all
        // slots and sums them in split order, so the result does not depend on arrival order.
        // PLM_MEASURE_SKIP_REDUCTION (a measurement build only, never the shipped library): the
        // split workgroups write their own partial sums as the result, so timing the same
        // launches with and without it gives the cost of the split-K reduction (wrong results).
#ifndef PLM_MEASURE_SKIP_REDUCTION
#define PLM_MEASURE_SKIP_REDUCTION 0
#endif
        if (!PERSIST && a.splits > 1 && !PLM_MEASURE_SKIP_REDUCTION) {
            constexpr int TILE_BYTES = MT * NS * NT * 16;
            const __amdgpu_buffer_rsrc_t p_rsrc = make_rsrc(
                reinterpret_cast<uint8_t*>(a.partial) + static_cast<int64_t>(blockIdx.x) * a.splits * TILE_BYTES,
                static_cast<uint32_t>(a.splits * TILE_BYTES));
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NS; ++j)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), p_rsrc,
                                                           ((i * NS + j) * NT + tid) * 16, split * TILE_BYTES, kCoherent);
            hold_until_stored(acc);
            if (!arrive_last(&a.counters[blockIdx.x], static_cast<uint32_t>(a.splits), &last_flag)) return;
            // Several splits' loads in flight where the registers allow (one at a time, each split
            // costs a memory round trip): SB of them, past the last one out of range.
            constexpr int SB = split_batch(MT, NS);
            for (int s0 = 0; s0 < a.splits; s0 += SB) {
                f32x4_t v[SB][MT][NS];
#pragma unroll
                for (int q = 0; q < SB; ++q) {
                    const bool in = s0 + q < a.splits;
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NS; ++j)
                            v[q][i][j] = __builtin_bit_cast(
                                f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                             p_rsrc, in ? ((i * NS + j) * NT + tid) * 16 : kOOB,
                                             in ? (s0 + q) * TILE_BYTES : 0, kCoherent));
                }
#pragma unroll
                for (int q = 0; q < SB; ++q)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NS; ++j)
                            acc[i][j] = s0 + q == 0 ? v[q][i][j] : acc[i][j] + v[q][i][j];
            }
        }

        epilogue(cur, acc, last_stage);
        if (!PERSIST || next < 0) return;
        cur = nxt;
        stage0 = last_stage ^ 1;
        loaded = true;
    }
}

// Tile shapes: {WM, WN, MT, NS}.
struct shape {
    int wm, wn, mt, ns;
    constexpr int bm() const { return wm * mt * 16; }
    constexpr int bs() const { return wn * ns; }
};
// The 256-row shapes take int4 weights or W8A8 (fp8 weight tiles staged in LDS beside bf16 x
// would not fit); kTall also takes fp8 W8A16, whose weight tiles then go to registers.
constexpr shape kHuge{2, 4, 8, 4};   // 256 x 256, 8 wavefronts (two stages fill the 160 KiB LDS)
constexpr shape kWide{2, 4, 8, 3};   // 256 x 192, 8 wavefronts (N = 6144 gives whole rounds)
constexpr shape kTall{1, 8, 16, 2};  // 256 x 256, 8 wavefronts of 256 x 32: each strip dequantized once
constexpr shape kTallHalf{1, 8, 8, 2};  // 128 x 256, 8 wavefronts of 128 x 32 (also kTall's tail launch)
constexpr shape kLarge{2, 2, 8, 4};  // 256 x 128, 4 wavefronts
constexpr shape kLarge8{2, 4, 8, 2};  // 256 x 128, 8 wavefronts of 128 x 32 (plain fp8 W8A16)
constexpr shape kSmall{2, 2, 4, 4};  // 128 x 128, 4 wavefronts
// One row of wavefronts on short tiles: each strip is dequantized once, as on kTall, with two
// workgroups on a CU. Against the shapes that share strips between wavefront rows: fp8 W8A16
// K 5120, N 7168, M = 333 74.8 -> 43.5 us, M = 2000 175 -> 147; int4 K 12288, N 4096, M = 333
// 72 -> 51, K 4096, N 6144, M = 800 65 -> 54; W8A8 K 5120, N 7168, M = 333 52 -> 36.
constexpr shape kOne128w4{1, 4, 8, 2};  // 128 x 128, 4 wavefronts of 128 x 32
constexpr shape kOne128w8{1, 8, 8, 1};  // 128 x 128, 8 wavefronts of 128 x 16
constexpr shape kOne96{1, 4, 6, 2};     // 96 x 128
constexpr shape kOne112{1, 4, 7, 2};    // 112 x 128
constexpr shape kOne96x256{1, 8, 6, 2};  // 96 x 256
// Grouped calls also use short row blocks for experts with few rows.
constexpr shape kRows16{1, 4, 1, 2};  // 16 x 128
constexpr shape kRows64{1, 4, 4, 2};  // 64 x 128
constexpr shape kRows64w8{1, 8, 4, 1};  // 64 x 128, 8 wavefronts of one strip (plain int4 calls)
constexpr shape kRows32{1, 4, 2, 2};  // 32 x 128 (grouped)

// Shapes of plain calls, and which modes have them.
enum shape_id { kIdS, kIdR, kIdW, kIdX, kIdQ, kIdG, kIdH, kIdA, kIdB, kIdC, kIdD, kIdF, kShapes };
constexpr char kShapeLetter[kShapes + 1] = "SRWXQGHABCDF";
constexpr shape kShapeOf[kShapes] = {kSmall,    kRows64,   kWide,     kTall,  kRows64w8, kLarge8,
                                     kTallHalf, kOne128w4, kOne128w8, kOne96, kOne112,   kOne96x256};
enum mfma_mode { kModeInt4, kModeFp8, kModeA8 };
// Bit i: shape i. The 256-row shapes with 12 or 16 strips need int4 weights or e4m3 x: with bf16 x
// and 2 KiB fp8 tiles two stages would not fit the 160 KiB LDS (kTall then keeps the weights in registers).
constexpr uint32_t kModeShapes[3] = {
    1u << kIdR | 1u << kIdW | 1u << kIdX | 1u << kIdQ | 1u << kIdH | 1u << kIdB | 1u << kIdC | 1u << kIdD | 1u << kIdF,
    1u << kIdR | 1u << kIdX | 1u << kIdG | 1u << kIdA | 1u << kIdB | 1u << kIdC | 1u << kIdD | 1u << kIdF,
    1u << kIdS | 1u << kIdR | 1u << kIdW | 1u << kIdX | 1u << kIdH | 1u << kIdA | 1u << kIdB | 1u << kIdC | 1u << kIdD};

// A plain launch of shape `id` (one of kModeShapes[the mode]).
template <plm_format F, bool BF16, bool UNIFORM, bool WIDE, bool A8, int I = 0>
void launch_shape(const mfma_args& a, int id, dim3 grid, hipStream_t s) {
    if constexpr (I < kShapes) {
        constexpr mfma_mode mode = A8 ? kModeA8 : (F == PLM_FP8 ? kModeFp8 : kModeInt4);
        if (id != I) return launch_shape<F, BF16, UNIFORM, WIDE, A8, I + 1>(a, id, grid, s);
        if constexpr ((kModeShapes[mode] >> I & 1) != 0) {
            constexpr shape sh = kShapeOf[I];
            if constexpr ((I == kIdX && mode != kModeFp8) || I == kIdH) {  // the 16-byte epilogue of the unsplit tall shapes
                if (a.splits == 1 && (a.n & 7) == 0 && aligned(a.y, 16)) {
                    mfma_kernel<F, BF16, UNIFORM, WIDE, A8, false, sh.wm, sh.wn, sh.mt, sh.ns, true>
                        <<<grid, sh.wm * sh.wn * 64, 0, s>>>(a);
                    return;
                }
            }
            mfma_kernel<F, BF16, UNIFORM, WIDE, A8, false, sh.wm, sh.wn, sh.mt, sh.ns><<<grid, sh.wm * sh.wn * 64, 0, s>>>(a);
        }
    }
}

}  // namespace

void launch_plain_int4(const mfma_args& a, bool bf16, bool uniform, int id, dim3 grid, hipStream_t s);
void launch_plain_fp8(const mfma_args& a, bool bf16, bool uniform, int id, dim3 grid, hipStream_t s);
void launch_plain_a8(const mfma_args& a, bool bf16, int id, dim3 grid, hipStream_t s);

inline void fill_common(mfma_args& a, const void* x, const void* w, const void* scale, plm_dtype scale_dtype, int64_t m,
                        int64_t n, int64_t k, int64_t block_n, int64_t group_size, void* y) {
    const layout_dims d = make_dims(n, k, block_n, group_size);
    a.x = static_cast<const uint16_t*>(x);
    a.w = static_cast<const uint8_t*>(w);
    a.scale = scale;
    a.y = static_cast<uint16_t*>(y);
    a.scale_dtype = scale_dtype;
    a.scale_cols = d.scale_cols;
    a.m = static_cast<int>(m);
    a.n = static_cast<int>(n);
    a.k = static_cast<int>(k);
    a.ktiles = static_cast<int>(d.ktiles);
    a.strips = static_cast<int>(d.strips);
    a.groups = static_cast<int>(d.groups);
    a.group_size = static_cast<int>(group_size);
    a.group_inv = 1.f / static_cast<float>(group_size / 16);
}

}  // namespace plm
