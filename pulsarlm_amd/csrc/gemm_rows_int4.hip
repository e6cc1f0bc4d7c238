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
    return cache.get(f, m, n, k, 0, [&] { return make_rows_plan(f, m, n, k); });
}

static int64_t rows_need(const rows_plan& p) {
    if (p.rb == 0 || p.splits <= 1) return 0;
    return kCounterBytes + static_cast<int64_t>(p.m_blocks) * p.n_blocks * p.splits * p.rb * p.sg * 1024;
}
// The rows kernel or the decode / MFMA kernels, by both sides' times at 1358 random layers (N = 128..40000,
// K = 256..28672, groups of 16 to 640 and every scale type) and 20 to 25 row counts each. What decides is
// how many strips a CU gets and how many K tiles there are: the rows kernel's start and epilogue are paid
// per round of its workgroups (one to four strips each), and below 16 K tiles its eight wavefronts have less than
// two each. Ratios below are rows / other kernel, means over the layers of a range. rr: the round-robin
// decode kernel takes the call.
bool use_rows(plm_format f, int64_t m, int64_t n, int64_t k, int64_t group_size, bool rr) {
    const tuning& t = knobs();
    if (t.rows_force) return true;
    if (t.rows_off || t.decode_max_m >= 0 || t.decode_sp > 0 || t.rr_sg > 0 || t.decode_no_xs || t.mfma_shape) return false;
    const int64_t strips = ceil_div(n, kTileN), kt = ceil_div(k, kTileK), cus = cu_count();
    const bool sub = group_size % kTileK != 0, fp8 = f == PLM_FP8;
    auto up_to = [&](int64_t per_cu) { return strips <= per_cu * cus; };
    // Against the MFMA kernel. Above 64 rows the weights are read once per row block: up to one strip
    // per CU 0.35-0.95, up to two 0.5-0.9 but 1.0-1.2 past 64 K tiles, beyond 1.1-2.
    if (m > 64) return up_to(1) || (up_to(2) && kt > 2 && kt <= 64);
    if (m > 32) {
        if (up_to(4)) {  // 0.4-0.95
            if (kt <= (fp8 ? 4 : 8)) return up_to(kt > 2 ? 3 : 2);  // past it 1.0-1.15
            return fp8 || m <= 48 || kt <= 64 || up_to(2) || !up_to(3);  // int4 else 1.04-1.2
        }
        if (m > 48) return false;  // 1.0-1.8
        if (fp8) return kt > 8 && kt <= 64;  // 0.83-0.99; below 1.0-1.3, above 1.0-1.15
        return !up_to(5) && (up_to(6) ? kt >= 16 && kt <= 32 : kt >= 24 && kt <= 64);  // 0.84-1.0; outside 1.0-1.5
    }
    // 17 to 32 rows: 0.5-0.95; with fewer K tiles and more strips 1.05-2 against the decode kernels,
    // which stop at 24 rows from four strips per CU on.
    if (m > 16) return kt > 16 || up_to(3) || (up_to(6) && kt > (m > 24 ? 4 : 8));
    // Against the decode kernels. Where the round-robin one applies it is 3-25 % faster, but for int4 above
    // 4 rows from five strips per CU on (0.7-1.0), and for fp8 (up to 4 rows 0.75-0.97, above 0.7-0.95 past
    // 1.5 strips per CU) only between one and 1.5 strips per CU, and up to 4 rows from four on.
    if (rr) {
        if (!fp8) return m > 4 && strips >= 5 * cus;
        return m <= 4 ? up_to(1) || (2 * strips > 3 * cus && strips < 4 * cus) : 2 * strips > 3 * cus;
    }
    // Against the split-K one.
    if (fp8) {
        if (kt <= 4) return false;  // 1.0-1.4
        if (kt <= 8) return up_to(1) || (m > 4 && up_to(2));  // 0.7-0.8; past it 1.05-1.3
        if (up_to(1)) return m > 4 || 2 * strips <= cus || kt <= 32 || kt > 96;  // 0.63-0.98; else 1.0-1.17
        if (2 * strips <= 3 * cus) return m > 4 || kt <= 16 || kt > (m > 2 ? 64 : 96);  // 0.64-0.97; else 1.0-1.15
        if (m <= 2) return m == 2 && kt > 96 && strips < 4 * cus;  // 0.88-0.91; else 1.0-1.2
        if (kt <= 16) return m > 4 && up_to(3);  // 0.65-0.98; past it 1.0-1.25
        if (kt <= 32) return m <= 4 ? up_to(2) : up_to(3) || (m > 8 && kt > 24);  // 0.8-0.99; past it 1.0-1.15
        return m <= 4 || m > 8 || up_to(4) || kt > 48;  // 0.75-0.99; past it 1.0-1.1
    }
    if (kt <= 4) return m > 4 && up_to(sub ? 6 : 1);  // 0.8-1.0; past it 1.05-1.4
    if (kt <= 8) return up_to(1) || (m > 4 && (up_to(3) || sub));  // 0.55-0.98; past it 1.0-1.3
    // Exactly one strip per CU over a K whose x the split-K kernel holds in LDS: it runs unsplit in one
    // round (K 13312, M = 1: 8.6 us against 9.5; K 20480, M = 2: 11.6 against 13.0). With fewer strips it
    // splits K, with more it takes a second round (K 13312, M = 1, N 4080: 12.1 against 9.8, N 4112: 13.7
    // against 11.2), and x from global memory costs it the lead (K 13312, M = 4: 11.5 against 9.7).
    if (!sub && strips == cus && m * k * 2 <= kStageMaxBytes && m <= kStageMaxM) return false;
    // 0.4-0.98, but groups of whole tiles at 17 to 32 K tiles 1.03-1.07 up to 2 rows.
    if (up_to(4)) return m > 2 || sub || kt <= 16 || kt > 32 || 2 * strips <= 3 * cus;
    // Past four strips per CU the split-K kernel takes two strips a wavefront: up to 2 rows 0.8-0.95 (N 18944,
    // K 4480, M = 1: 13.3 us against 13.7; K 6144: 16.2 against 17.1), up to 4 (x of 3 rows and more
    // costs it a quarter past 32 K tiles) and 8 rows 0.85-0.97 against the rows kernel outside these.
    if (m <= 2) return sub ? kt <= 16 || kt > 48 : kt > (m == 1 ? 96 : 64);
    if (m <= 4) return kt > 32 || (sub && kt <= 16);
    return sub || m > 8 || kt > 48;
}

// For calls of a size: no group size or scale layout, so what any of them may need.
int64_t rows_workspace_bytes(plm_format f, int64_t m, int64_t n, int64_t k) {
    if (m > kRowsMaxM) return 0;
    const bool any = use_rows(f, m, n, k, kTileK, false) || use_rows(f, m, n, k, kTileK, true) ||
                     (f == PLM_INT4 && use_rows(f, m, n, k, kTileK / 2, false));
    return any ? rows_need(plan_rows(f, m, n, k)) : 0;
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
    c.taken = c.lds <= 160 * 1024;  // the plan does not look at the scales: 32-wide groups over a long K may not fit
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
