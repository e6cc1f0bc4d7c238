// Dequant-GEMM for decode batches and short prefills (up to 128 rows):
// y[M, N] = x[M, K] @ dequant(W)^T.
//
// A workgroup owns RB blocks of 16 rows by SG strips of 16 columns over one K range; its
// eight wavefronts take the range's 128-wide K tiles round-robin, so a wavefront holds all
// RB x SG accumulators of its own K tiles and nothing is shared before the end:
// * every x value is read from LDS by one wavefront only and feeds SG MFMAs. With the
//   wavefronts side by side on the columns (gemm_mfma.hip) each reads the whole x tile, and at
//   these sizes that kernel spends its time on the barrier of every K step, the x fragment
//   reads and a serial chain of short steps; staging three to six K steps ahead of it gained
//   3 % (M = 48, K = N = 4096: 11.5 us, whose weights stream in 1.7 us);
// * x half tiles (64 K, 128 bytes a row: whole cache lines) go to the wavefront's own ring of D
//   slots with buffer loads to LDS, the weights of the next K tile to registers; the
//   wavefront waits for its own loads by count, and no barrier stands in the K loop;
// * the scales of the K range are staged once at the start;
// * the wavefronts' sums are added through LDS in wavefront order, K ranges of different
//   workgroups by the last one to arrive, in split order: deterministic.
// What bounds it: the x bytes a CU pulls from L2 (RB x 16 x K x 2 per workgroup, about 85 B/ns
// a CU with these copies; 16-byte gathers of MFMA fragments straight to registers reached a
// third of that), then the dequant and MFMA issue of two to four wavefronts per SIMD.
// Measured against the kernels it replaces (MI355X, graph replays over cold weights, us):
//   int4 g128         M = 32            M = 48            M = 64
//   K 4096,  N 4096    9.2 ->  6.7      11.5 ->  8.1      11.8 ->  9.1
//   K 4096,  N 6144   10.5 ->  8.0      12.4 ->  9.7      12.8 -> 11.2
//   K 4096,  N 24576  26.4 -> 17.6      27.3 -> 24.2      28.0 -> 27.3
//   K 12288, N 4096   15.4 -> 12.7      18.6 -> 14.4      19.0 -> 16.3
//   fp8 K 5120, N 34816: M = 16 43.0 -> 33.2, M = 32 78.1 -> 40.4, M = 64 79.5 -> 56.4
//   fp8 K 17408, N 5120: M = 4 28.0 -> 19.8, M = 16 28.1 -> 20.1, M = 64 40.5 -> 28.9
#pragma once

#include "plm_common.hpp"

namespace plm {

struct rows_args {
    const uint16_t* x;
    const uint8_t* w;
    const uint8_t* scale;
    uint16_t* y;
    float* partial;
    uint32_t* counters;
    int m, n, k;
    int ktiles, strips, groups;
    int splits, tiles_per_split;
    int m_blocks;
    int scale_dtype;
    uint32_t group_magic;  // k / group_size = umulhi(2 (k / 16), group_magic)
    int s_stage;           // staged scale bytes per strip, a multiple of 256
};

// Tile shapes. Slots of the x ring: as many as leave LDS for two workgroups on a CU up to 32
// rows (64 KiB of x each); above, two slots fill one workgroup's share.
constexpr int kRowsWaves = 8;
constexpr int rows_slots(int rb) { return rb == 1 ? 4 : 2; }
constexpr int rows_red_blocks(int rb, int sg) { return rb * sg <= 20 ? rb : 20 / sg; }  // row blocks per LDS reduction pass
constexpr int64_t rows_lds_bytes(int rb, int sg, int64_t s_stage) {
    const int64_t loop = sg * s_stage + int64_t{kRowsWaves} * rows_slots(rb) * rb * 2048;
    const int64_t red = int64_t{rows_red_blocks(rb, sg)} * sg * kRowsWaves * 1024;
    return loop > red ? loop : red;
}

// SCM: scale layout per (strip, group): 0 = 16 x 16-bit, 1 = 16 x fp32, 2 = 1 x fp32.
// SUB: group_size is not a multiple of 128 (scales looked up per 32-wide K slice and lane).
template <plm_format F, bool BF16, int SCM, bool SUB, int RB, int SG>
__global__ void __launch_bounds__(kRowsWaves * 64) rows_kernel(rows_args a) {
    constexpr int NW = kRowsWaves;
    constexpr int TB = fmt_traits<F>::tile_bytes;
    constexpr int NL = TB / 1024;
    constexpr bool WIDE = SCM != 0;
    constexpr int ES = WIDE ? 4 : 2;
    constexpr int EB = (SCM == 2 ? 1 : 16) * ES;  // scale bytes per (strip, group)
    constexpr int D = rows_slots(RB);
    constexpr int XL = RB * 2;       // x copies per half tile
    constexpr int WL = SG * NL;      // weight loads per K tile
    constexpr int SLOT = RB * 2048;  // bytes of an x half tile
    extern __shared__ __attribute__((aligned(16))) uint8_t rows_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int col16 = lane & 15, kq = lane >> 4;
    const bool bf16_scale = a.scale_dtype == PLM_BF16;

    const int tile = blockIdx.x, split = blockIdx.y;
    const int strip0 = tile / a.m_blocks * SG, row0 = (tile % a.m_blocks) * RB * 16;
    const int rows = min(RB * 16, a.m - row0);
    const int kt_lo = split * a.tiles_per_split;
    const int kt_hi = min(kt_lo + a.tiles_per_split, a.ktiles);
    auto group_of = [&](int k) { return static_cast<int>(__umulhi(static_cast<uint32_t>(k >> 4) << 1, a.group_magic)); };

    // The scales of the K range, [strip][group][EB]; strips past N read zeros.
    const int g_lo = group_of(kt_lo * kTileK);
    {
        const __amdgpu_buffer_rsrc_t sr = make_rsrc(a.scale, static_cast<uint32_t>(a.strips) * a.groups * EB);
        const int have = (a.groups - g_lo) * EB;
        for (int o = wave * 256; o < SG * a.s_stage; o += NW * 256) {  // wave-uniform
            const int sj = o / a.s_stage, in = o - sj * a.s_stage + lane * 4;
            const int st = strip0 + sj;
            const int off = st < a.strips && in < have ? (st * a.groups + g_lo) * EB + in : kOOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (__attribute__((address_space(3))) void*)(rows_lds + o), 4, off, 0, 0, 0);
        }
    }

    const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x + static_cast<int64_t>(row0) * a.k, static_cast<uint32_t>(rows) * a.k * 2);
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.w, static_cast<uint32_t>(a.strips) * a.ktiles * TB);
    int w_strip[SG];  // tile index of each strip's first K tile; strips past N reload the last one (never stored)
#pragma unroll
    for (int sj = 0; sj < SG; ++sj) w_strip[sj] = min(strip0 + sj, a.strips - 1) * a.ktiles;
    // A copy is 8 rows x 128 bytes; the 16-byte columns are XOR-swizzled by row, so that the 16
    // rows of a fragment read fall in different banks.
    uint8_t* xs = rows_lds + SG * a.s_stage + wave * (D * SLOT);
    int x_off[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = i * 8 + (lane >> 3);
        x_off[i] = r * a.k * 2 + (((lane & 7) ^ (r & 7)) << 4);  // rows past `rows` are past the buffer's end
    }
    const int w_lane = lane * 16;

    struct wbatch {
        u32x4_t w[SG][NL];
    };
    auto load_w = [&](wbatch& b, int kt) {
        const int past = kt < kt_hi ? 0 : kOOB;
#pragma unroll
        for (int sj = 0; sj < SG; ++sj)
#pragma unroll
            for (int h = 0; h < NL; ++h)
                b.w[sj][h] = buffer_load16_stream(wr, (w_lane + h * 1024) | past, past ? 0 : (w_strip[sj] + kt) * TB);
    };
    auto load_x = [&](int kt, int h, int slot) {
        const int past = kt < kt_hi ? 0 : kOOB;
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            int off = x_off[i] | past;
            if constexpr (SUB)  // K may end inside the last tile
                off |= kt * 256 + h * 128 + (((lane & 7) ^ (lane >> 3)) << 4) >= a.k * 2 ? kOOB : 0;
            buffer_load_lds16(xr, xs + slot * SLOT + i * 1024, off, past ? 0 : kt * 256 + h * 128);
        }
    };

    f32x4_t acc[RB][SG];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int sj = 0; sj < SG; ++sj) acc[rb][sj] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    struct scales {
        int4_scale k4[SG];
        float s8[SG];
    };
    auto set_scale = [&](scales& s, int sj, int k) {
        const uint8_t* p = rows_lds + sj * a.s_stage + (group_of(k) - g_lo) * EB + (SCM == 2 ? 0 : col16 * ES);
        const uint32_t bits = WIDE ? *reinterpret_cast<const uint32_t*>(p)
                                   : static_cast<uint32_t>(*reinterpret_cast<const uint16_t*>(p));
        const float raw = scale_from_bits<WIDE>(bits, bf16_scale);
        if constexpr (F == PLM_INT4) s.k4[sj] = make_int4_scale<BF16>(raw);
        else s.s8[sj] = round_to<BF16>(raw);
    };

    int slot = 0;
    // Half h of K tile kt: requests the half tile D - 1 ahead (of tile kt + NW * (...)) into the
    // slot read last, waits for its own, and multiplies. Issue order: ... x(h), x(h + 1), ..; the
    // next tile's weights before the first half's request. So after x(h) come D - 1 halves and,
    // except for the second half with two slots, one tile's weights.
    auto half = [&](const wbatch& b, int kt, int h, scales& s) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's reads of that slot
        load_x(kt + NW * ((h + D - 1) >> 1), (h + D - 1) & 1, slot == 0 ? D - 1 : slot - 1);
        if (D == 2 && h == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * XL) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * XL + WL) : "memory");
        const uint8_t* sx = xs + slot * SLOT;
        slot = slot == D - 1 ? 0 : slot + 1;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const int t = 2 * h + tt;
            u32x4_t x[RB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                x[rb] = *reinterpret_cast<const u32x4_t*>(sx + (16 * rb + col16) * 128 + (((4 * tt + kq) ^ (col16 & 7)) << 4));
#pragma unroll
            for (int sj = 0; sj < SG; ++sj) {
                if constexpr (SUB) set_scale(s, sj, kt * kTileK + 32 * t + 8 * kq);
                u32x4_t bop;
                if constexpr (F == PLM_INT4) bop = dq_int4<BF16>(b.w[sj][0][t], s.k4[sj]);
                else bop = dq_fp8<BF16>(b.w[sj][t >> 1][(t & 1) * 2], b.w[sj][t >> 1][(t & 1) * 2 + 1], s.s8[sj]);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) acc[rb][sj] = mfma16x16x32<BF16>(x[rb], bop, acc[rb][sj]);
            }
        }
    };
    auto k_tile = [&](const wbatch& b, wbatch& next, int kt) {
        load_w(next, kt + NW);
        scales s;
        if constexpr (!SUB) {
#pragma unroll
            for (int sj = 0; sj < SG; ++sj) set_scale(s, sj, kt * kTileK);
        }
        half(b, kt, 0, s);
        half(b, kt, 1, s);
    };

    const int first = kt_lo + wave;
    wbatch w0, w1;
    load_w(w0, first);
#pragma unroll
    for (int h = 0; h < D - 1; ++h) load_x(first + NW * (h >> 1), h & 1, h);
    // Every wavefront's share of the scales (requested before these loads) has landed.
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WL + (D - 1) * XL) : "memory");
    for (int kt = first; kt < kt_hi; kt += 2 * NW) {
        k_tile(w0, w1, kt);
        if (kt + NW >= kt_hi) break;
        k_tile(w1, w0, kt + NW);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // requests past the last tile

    // Sums over the wavefronts through LDS, in wavefront order, PER row blocks at a time. Unit u
    // is 16 bytes of the output tile: rows 16 rb + 4 (ln / 16) .. + 3 of column ln % 16 of strip sj.
    constexpr int PER = rows_red_blocks(RB, SG);
    constexpr int UNITS = RB * SG * 64;
    f32x4_t* red = reinterpret_cast<f32x4_t*>(rows_lds);
    const __amdgpu_buffer_rsrc_t pr =
        make_rsrc(reinterpret_cast<uint8_t*>(a.partial) + static_cast<int64_t>(tile) * a.splits * UNITS * 16,
                  a.splits > 1 ? static_cast<uint32_t>(a.splits) * UNITS * 16 : 0u);
    auto store_unit = [&](int u, const f32x4_t& v) {
        const int ln = u & 63, rb = (u >> 6) / SG, sj = (u >> 6) % SG;
        const int col = (strip0 + sj) * kTileN + (ln & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * rb + 4 * (ln >> 4) + i;
            if (r < rows && col < a.n)
                a.y[static_cast<int64_t>(row0 + r) * a.n + col] = static_cast<uint16_t>(to_bits16<BF16>(v[i]));
        }
    };
#pragma unroll
    for (int rb0 = 0; rb0 < RB; rb0 += PER) {
        const int blocks = rb0 + PER < RB ? PER : RB - rb0;
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < PER; ++rb)
            if (rb0 + rb < RB) {
#pragma unroll
                for (int sj = 0; sj < SG; ++sj) red[((rb * SG + sj) * NW + wave) * 64 + lane] = acc[rb0 + rb][sj];
            }
        __syncthreads();
        constexpr int ITERS = (PER * SG * 64 + NW * 64 - 1) / (NW * 64);
        f32x4_t v[ITERS][1];
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int q = threadIdx.x + it * NW * 64;
            if (q >= blocks * SG * 64) continue;
            const f32x4_t* p = red + (q >> 6) * NW * 64 + (q & 63);
            v[it][0] = p[0];
#pragma unroll
            for (int w = 1; w < NW; ++w) v[it][0] = v[it][0] + p[w * 64];
            const int u = rb0 * SG * 64 + q;
            if (a.splits == 1) store_unit(u, v[it][0]);
            else
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v[it][0]), pr, u * 16, split * UNITS * 16,
                                                       kCoherent);
        }
        if (a.splits > 1) hold_until_stored(v);
    }
    if (a.splits == 1) return;
    if (!arrive_last(&a.counters[tile], static_cast<uint32_t>(a.splits), reinterpret_cast<uint32_t*>(rows_lds))) return;
    for (int u = threadIdx.x; u < UNITS; u += NW * 64) {
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < a.splits; s0 += 4) {  // four splits' loads in flight
            f32x4_t p[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                p[q] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                       pr, s0 + q < a.splits ? u * 16 : kOOB,
                                                       s0 + q < a.splits ? (s0 + q) * UNITS * 16 : 0, kCoherent));
#pragma unroll
            for (int q = 0; q < 4; ++q) v = v + p[q];
        }
        store_unit(u, v);
    }
}

// Launches shape (rb, sg) for the format in F; false where it has no instantiation.
template <plm_format F> bool launch_rows_shape(const rows_args& a, bool bf16, int scm, bool sub, int rb, int sg, dim3 grid,
                                               size_t lds, hipStream_t s);

}  // namespace plm
