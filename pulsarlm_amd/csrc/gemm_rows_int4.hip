// rows_kernel for int4 weights, and the plan and launch of rows calls.
#include <algorithm>
#include <type_traits>

#include "gemm_rows.hpp"

namespace plm {

bool decode_rr_takes(plm_format f, int64_t m, int64_t n, int64_t k, int64_t block_n, int64_t group_size, plm_dtype scale_dtype);

namespace {

template <bool BF16, int SCM, bool SUB, int RB, int SG>
void launch_one(const rows_args& a, dim3 grid, size_t lds, hipStream_t s) {
    rows_kernel<PLM_INT4, BF16, SCM, SUB, RB, SG><<<grid, kRowsWaves * 64, lds, s>>>(a);
}

template <bool BF16, int SCM, bool SUB, int RB>
bool launch_sg(const rows_args& a, int sg, dim3 grid, size_t lds, hipStream_t s) {
    switch (sg) {
        case 1: launch_one<BF16, SCM, SUB, RB, 1>(a, grid, lds, s); return true;
        case 2: launch_one<BF16, SCM, SUB, RB, 2>(a, grid, lds, s); return true;
        case 3: launch_one<BF16, SCM, SUB, RB, 3>(a, grid, lds, s); return true;
        case 4: launch_one<BF16, SCM, SUB, RB, 4>(a, grid, lds, s); return true;
        default: return false;
    }
}

template <bool BF16, int SCM, bool SUB>
bool launch_rb(const rows_args& a, int rb, int sg, dim3 grid, size_t lds, hipStream_t s) {
    switch (rb) {
        case 1: return launch_sg<BF16, SCM, SUB, 1>(a, sg, grid, lds, s);
        case 2: return launch_sg<BF16, SCM, SUB, 2>(a, sg, grid, lds, s);
        case 3: return launch_sg<BF16, SCM, SUB, 3>(a, sg, grid, lds, s);
        case 4: return launch_sg<BF16, SCM, SUB, 4>(a, sg, grid, lds, s);
        default: return false;
    }
}

template <typename Fn> bool dispatch(bool bf16, int scm, bool sub, Fn fn) {
    if (scm != 0 && scm != 1) return false;
    const int mode = (bf16 ? 4 : 0) + (scm ? 2 : 0) + (sub ? 1 : 0);
    switch (mode) {
        case 0: return fn(std::false_type{}, std::integral_constant<int, 0>{}, std::false_type{});
        case 1: return fn(std::false_type{}, std::integral_constant<int, 0>{}, std::true_type{});
        case 2: return fn(std::false_type{}, std::integral_constant<int, 1>{}, std::false_type{});
        case 3: return fn(std::false_type{}, std::integral_constant<int, 1>{}, std::true_type{});
        case 4: return fn(std::true_type{}, std::integral_constant<int, 0>{}, std::false_type{});
        case 5: return fn(std::true_type{}, std::integral_constant<int, 0>{}, std::true_type{});
        case 6: return fn(std::true_type{}, std::integral_constant<int, 1>{}, std::false_type{});
        default: return fn(std::true_type{}, std::integral_constant<int, 1>{}, std::true_type{});
    }
}

}  // namespace

template <>
bool launch_rows_shape<PLM_INT4>(const rows_args& a, bool bf16, int scm, bool sub, int rb, int sg, dim3 grid, size_t lds,
                                 hipStream_t s) {
    return dispatch(bf16, scm, sub, [&](auto b, auto c, auto u) { return launch_rb<b.value, c.value, u.value>(a, rb, sg, grid, lds, s); });
}

// Which plain calls the rows kernel takes, with which tile and K split. The time of a tile is the
// x it copies, the weights it dequantizes and multiplies, and a start; the workgroups run in
// rounds over the CUs (a last round that is partly full costs nearly a whole one); a K split
// adds the exchange of partial sums. The constants (us; per 128-wide K tile) are a fit to 1300
// timings, each shape and split at nine int4 and seven fp8 layers (K = 2048..17408, N = 1024..
// 34816) and eight row counts from 5 to 128; over them the pick is 0.6 % (int4) and 0.9 % (fp8)
// slower than the best shape.
struct rows_plan {
    int rb = 0, sg = 0;  // rb == 0: not taken
    int m_blocks = 0, n_blocks = 0, splits = 0, tiles_per_split = 0;
};

constexpr int64_t kRowsMaxM = 128;
constexpr int64_t kRowsMaxK = int64_t{1} << 19;  // group lookup by reciprocal: K / 16 times group_size / 16 below 2^31
constexpr int64_t kRowsMaxPartials = 24 << 20;   // with the counters, within plm_gemm_noalloc's fixed scratch

struct rows_cost {
    double x, w[4], start, last_round, split, split_tile, split_each;
};
constexpr rows_cost kRowsInt4{0.0332, {0.0414, 0.0464, 0.0641, 0.0697}, 0.864, 0.812, 0.286, 0.161, 0.279};
constexpr rows_cost kRowsFp8{0.0402, {0.0641, 0.0692, 0.0847, 0.0855}, 0.873, 0.871, 0.412, 0.180, 0.281};

rows_plan make_rows_plan(plm_format f, int64_t m, int64_t n, int64_t k) {
    rows_plan best;
    const int64_t strips = ceil_div(n, kTileN), ktiles = ceil_div(k, kTileK), cus = cu_count();
    if (strips * ktiles * tile_bytes(f) >= kOOB) return best;
    const int64_t m_blocks = ceil_div(m, 64);  // above 64 rows: two row blocks
    const int rb = static_cast<int>(ceil_div(ceil_div(m, m_blocks), 16));
    const rows_cost& c = f == PLM_INT4 ? kRowsInt4 : kRowsFp8;
    double least = 0;
    const int kt = static_cast<int>(ktiles), mb = static_cast<int>(m_blocks), nc = static_cast<int>(cus);
    for (int sg = 1; sg <= 4; ++sg) {
        if (knobs().rows_sg > 0 && sg != knobs().rows_sg) continue;  // PLM_ROWS="sg,splits" (tuning sweeps)
        const int n_blocks = (static_cast<int>(strips) + sg - 1) / sg;
        const int64_t wgs = m_blocks * n_blocks;
        for (int want = 1; want <= std::min(8, kt); ++want) {
            const int tps = (kt + want - 1) / want, splits = (kt + tps - 1) / tps;
            if (splits != want || (knobs().rows_splits > 0 && splits != knobs().rows_splits)) continue;
            // Past two rounds a further split never pays.
            if (splits > 1 && (wgs * (splits - 1) >= 2 * cus || wgs > kMaxCounters ||
                               wgs * splits * rb * sg * 1024 > kRowsMaxPartials))
                break;
            const int all = static_cast<int>(wgs) * splits;
            const double full = static_cast<double>(all) / nc;
            const double rounds = full <= 1.0 ? 1.0 : full + c.last_round * ((all + nc - 1) / nc - full);
            const double t = rounds * (tps * (rb * c.x + sg * c.w[rb - 1]) + c.start) +
                             (splits > 1 ? c.split + c.split_tile * rb * sg + c.split_each * splits : 0.0);
            if (best.rb == 0 || t < least) {
                least = t;
                best.rb = rb, best.sg = sg;
                best.m_blocks = mb, best.n_blocks = n_blocks;
                best.splits = splits, best.tiles_per_split = tps;
            }
        }
    }
    return best;
}

rows_plan plan_rows(plm_format f, int64_t m, int64_t n, int64_t k) {
    if (m < 1 || m > kRowsMaxM || k > kRowsMaxK || n > (int64_t{1} << 24)) return rows_plan{};
    thread_local plan_cache<rows_plan> cache;
    return cache.get(f, m, n, k, [&] { return make_rows_plan(f, m, n, k); });
}

static int64_t rows_need(const rows_plan& p) {
    if (p.rb == 0 || p.splits <= 1) return 0;
    return kCounterBytes + static_cast<int64_t>(p.m_blocks) * p.n_blocks * p.splits * p.rb * p.sg * 1024;
}
int64_t rows_workspace_bytes(plm_format f, int64_t m, int64_t n, int64_t k) { return rows_need(plan_rows(f, m, n, k)); }

// The rows kernel or the decode / MFMA kernels, by both sides' times at the layers above and at 31
// random ones (hidden 2048..5120, M = 1..128; us, without -> with the rows kernel). rr: the
// round-robin decode kernel takes the call.
// * 17 to 64 rows: the rows kernel (against the MFMA kernel int4 1.1-2.0x, fp8 1.01-1.8x), but int4
//   above 32 rows with more than four strips per CU, where the MFMA kernel is even or faster (K 4736,
//   N 21248, M = 64: 28.6 -> 32.7) unless three-strip tiles nearly fill whole rounds of the CUs and there
//   are at most 48 rows (K 5120, N 23040: M = 36 31.0 -> 29.3, M = 48 30.5 -> 30.7).
// * Above 64 the weights are read once per row block: up to two strips per CU and K = 8448 (int4
//   K 4736, N 5248, M = 96: 19.4 -> 15.0, K 8192, N 2432, M = 128: 16.2 -> 15.4; fp8 K 2944, N 3968, M = 128:
//   18.8 -> 11.0; beyond: int4 K 2048, N 8704, M = 96 14.3 -> 15.2, K 9088, N 3200, M = 112 21.8 -> 24.8).
// * Up to 16 rows int4: the round-robin kernel where it applies (3-8 % faster), but above 4 rows
//   with five strips or more per CU (K 4096, N 24576, M = 16: 15.4 -> 14.6). Elsewhere (long K,
//   groups below 128) the rows kernel (K 14336, N 5120, M = 1: 14.9 -> 12.3; K 8192, N 8192: 12.3 -> 9.6), but
//   up to 4 rows exactly one strip per CU over a K that the split-K decode kernel holds in three
//   load batches a wavefront (K 12288, N 4096: 8.1 against 9.3 at best; K 13312: 11.6 -> 9.7), and up
//   to 2 rows groups below 128 with four strips or more per CU (K 4992, N 24832: 25.9 -> 28.5).
// * Up to 16 rows fp8: the rows kernel, but the round-robin one with four strips or more per CU
//   up to 4 rows (K 3968, N 25600: 19.2 -> 23.4) and the split-K one up to 2 rows where that one does
//   not apply (K 4864, N 32768: 28.7 -> 30.6); and between one and 1.5 strips per CU, or up to one
//   above 4 rows, up to K = 5120 (even to 9 % slower); and up to 2 rows the split-K one at long K and
//   at most one strip per CU (K 12800, N 3968: 12.6 -> 13.7).
bool use_rows(plm_format f, int64_t m, int64_t n, int64_t k, int64_t group_size, bool rr) {
    const tuning& t = knobs();
    if (t.rows_force) return true;
    if (t.rows_off || t.decode_max_m >= 0 || t.decode_sp > 0 || t.rr_sg > 0 || t.decode_no_xs || t.mfma_shape) return false;
    const int64_t strips = ceil_div(n, kTileN), cus = cu_count();
    const bool sub = group_size % kTileK != 0;
    if (m > 64) return strips <= 2 * cus && k <= 66 * kTileK;
    if (m > 16) {
        const int64_t tiles3 = ceil_div(strips, 3);
        return f == PLM_FP8 || m <= 32 || strips <= 4 * cus || (m <= 48 && 10 * tiles3 >= 9 * round_up(tiles3, cus));
    }
    if (f == PLM_FP8) {
        if (strips >= 4 * cus && m <= (rr ? 4 : 2)) return false;
        if (strips <= cus) return m <= 4 ? rr || m > 2 : !(rr || k <= 5120);
        return 2 * strips > 3 * cus || !(rr || k <= 5120);
    }
    if (rr) return m > 4 && strips >= 5 * cus;
    if (sub) return m > 2 || strips < 4 * cus;
    return m > 4 || strips != cus || k > 12288;
}

// A call as the rows kernel would run it; `taken` is false where it does not take the call (the
// workspace aside, which launch_rows looks at).
struct rows_call {
    bool taken = false;
    rows_plan p;
    layout_dims d;
    int scm;
    int64_t s_stage, lds;
};

rows_call resolve_rows(plm_format f, plm_dtype scale_dtype, int64_t m, int64_t n, int64_t k, int64_t block_n, int64_t group_size) {
    rows_call c;
    const bool sub = group_size % kTileK != 0;
    if (m > kRowsMaxM || k > kRowsMaxK || (f == PLM_FP8 && sub) ||
        !use_rows(f, m, n, k, group_size, decode_rr_takes(f, m, n, k, block_n, group_size, scale_dtype)))
        return c;
    c.p = plan_rows(f, m, n, k);
    if (c.p.rb == 0) return c;
    c.d = make_dims(n, k, block_n, group_size);
    c.scm = c.d.scale_cols == 16 ? (scale_dtype == PLM_FP32 ? 1 : 0) : (scale_dtype == PLM_FP32 ? 2 : -1);
    if (f == PLM_INT4 ? c.scm != 0 && c.scm != 1 : c.scm != 1 && c.scm != 2) return c;  // no instantiation
    const int64_t eb = c.d.scale_cols * dtype_size(scale_dtype);
    if (c.d.strips * c.d.groups * eb >= kOOB) return c;
    const int64_t span = c.p.splits == 1 ? c.d.groups
                                         : std::min<int64_t>(c.d.groups, ceil_div(int64_t{c.p.tiles_per_split} * kTileK, group_size) + 1);
    c.s_stage = round_up(span * eb, 256);
    c.lds = rows_lds_bytes(c.p.rb, c.p.sg, c.s_stage);
    c.taken = c.lds <= 160 * 1024;
    return c;
}

// Returns false, with nothing launched, where the rows kernel does not take the call.
bool launch_rows(plm_format f, const void* x, bool bf16, const void* w, const void* scale, plm_dtype scale_dtype, int64_t m,
                 int64_t n, int64_t k, int64_t block_n, int64_t group_size, void* y, void* workspace, size_t workspace_bytes,
                 hipStream_t s) {
    const rows_call c = resolve_rows(f, scale_dtype, m, n, k, block_n, group_size);
    if (!c.taken) return false;
    const rows_plan& p = c.p;
    const layout_dims& d = c.d;
    const int64_t need = rows_need(p);
    if (need > 0 && (workspace == nullptr || static_cast<int64_t>(workspace_bytes) < need)) return false;
    rows_args a{};
    a.x = static_cast<const uint16_t*>(x);
    a.w = static_cast<const uint8_t*>(w);
    a.scale = static_cast<const uint8_t*>(scale);
    a.y = static_cast<uint16_t*>(y);
    a.counters = static_cast<uint32_t*>(workspace);
    a.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + kCounterBytes);
    a.m = static_cast<int>(m), a.n = static_cast<int>(n), a.k = static_cast<int>(k);
    a.ktiles = static_cast<int>(d.ktiles), a.strips = static_cast<int>(d.strips), a.groups = static_cast<int>(d.groups);
    a.splits = p.splits, a.tiles_per_split = p.tiles_per_split;
    a.m_blocks = p.m_blocks;
    a.scale_dtype = scale_dtype;
    const uint64_t g16 = static_cast<uint64_t>(group_size) / 16;
    a.group_magic = static_cast<uint32_t>(((uint64_t{1} << 31) + g16 - 1) / g16);
    a.s_stage = static_cast<int>(c.s_stage);
    const dim3 grid(static_cast<unsigned>(p.m_blocks * p.n_blocks), static_cast<unsigned>(p.splits));
    const bool sub = group_size % kTileK != 0;
    return f == PLM_INT4 ? launch_rows_shape<PLM_INT4>(a, bf16, c.scm, sub, p.rb, p.sg, grid, static_cast<size_t>(c.lds), s)
                         : launch_rows_shape<PLM_FP8>(a, bf16, c.scm, sub, p.rb, p.sg, grid, static_cast<size_t>(c.lds), s);
}

}  // namespace plm

extern "C" {
// Not part of the public ABI (include/pulsarlm_amd.h): how plm_gemm would run a call on the rows kernel
// given enough workspace, for the tests that aim at it. out[0..5]: taken (0/1), row blocks and strips
// of a workgroup, workgroups over rows and columns, K splits.
__attribute__((visibility("default"))) void plm_internal_rows_plan(int format, int64_t m, int64_t n, int64_t k, int64_t block_n,
                                                                  int64_t group_size, int scale_dtype, int32_t* out) {
    using namespace plm;
    const rows_call c = resolve_rows(static_cast<plm_format>(format), static_cast<plm_dtype>(scale_dtype), m, n, k, block_n, group_size);
    out[0] = c.taken ? 1 : 0;
    out[1] = c.p.rb, out[2] = c.p.sg;
    out[3] = c.p.m_blocks, out[4] = c.p.n_blocks;
    out[5] = c.p.splits;
}
}  // extern "C"
