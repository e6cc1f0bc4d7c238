// Plans and launches of the MFMA kernel for plain and W8A8 calls.
#include <algorithm>
#include <cmath>

#include "gemm_mfma.hpp"

namespace plm {

struct mfma_config {
    int shape = -1;  // shape_id
    int m_blocks = 0, n_blocks = 0;
    int splits = 1, tiles_per_split = 0;
    // kTall only: the tiles past whole rounds of the CUs run as a second launch, as 128-row halves of
    // whole columns of tiles (halves), or with K split, so that the last round is shorter.
    int tail_tiles = 0, tail_splits = 0, tail_tiles_per_split = 0;
    bool tail_halves = false;
    int64_t need = 0;  // workspace bytes
};

// Estimated time of a shape and K split: the K steps of the workgroups a CU gets (co-resident ones
// share it: two cost less than twice one) with a start of `fill` steps, bounded below by the tile
// bytes that come through L2; a K split adds the exchange of its partial sums. The constants are
// a fit to 2600 timings: each shape and split at six layers (K = 2048..12288, N = 2048..14336) and
// nine row counts from 136 to 3300. Over them the pick is 1.3 % (int4) and 1.4 % (fp8) slower than the best
// shape. W8A8 is a fit to 7480 timings at 263 random sizes (M = 33..6000, N = 960..35200, K = 1024..19200), 1.5 %
// off the best there and 1.4 % at 87 others; with the constants from the six layers 6.9 and 4.9 %, at
// worst 1.6 times (a start of six K tiles on the 64-row shape sent short calls to others: M = 236, N = 1568,
// K = 2944 21.7 -> 15.0 us). The rule before it counted whole rounds of K tiles times the tile area
// over one rate a shape and had no tile heights of 96 and 112 rows: int4 M = 333, N = 6144, K = 4096
// 36.3 -> 27.5 us, fp8 M = 1000, N = 7168, K = 5120 107 -> 79, W8A8 M = 2048, N = 5120, K = 17408
// 240 -> 219.
struct shape_cost {
    // us per K tile with one, two and three workgroups on a CU. 0: LDS or registers hold no more, and a
    // further one waits (fp8 D has two: 186 VGPRs and twice 57 KiB; with a joint rate for three it was picked at
    // 15-25 % below its time: fp8 M = 402, N = 33888, K = 2688 118.7 us on D, 99.9 on C).
    double step[3];
    double fill;     // K tiles
};
struct mode_cost {
    double launch;      // us
    double reduce;      // us a K split
    double reduce_pass;  // us more for each further pass of the last workgroup over the splits
    double reduce_mib;  // us per MiB of partial sums
    double memory;      // us per MB of x and weight tiles
    shape_cost shapes[kShapes];  // in shape_id order
};
constexpr mode_cost kModeCost[3] = {
    // int4: -, R, W, X, Q, -, H, -, B, C, D, F
    {3.64, 2.09, 0, 0.185, 0.0907,
     {{}, {{0.7425, 1.0481, 1.4028}, 1.29}, {{2.6043, 0, 0}, 2.58}, {{2.6513, 0, 0}, 2.62}, {{0.6862, 1.0969, 0}, 0.85}, {},
      {{1.5961, 0, 0}, 3.18}, {}, {{0.9172, 1.8354, 0}, 2.78}, {{1.0175, 1.3798, 0}, 1.59}, {{1.1135, 1.4712, 0}, 2.47},
      {{1.3813, 2.8355, 0}, 3.20}}},
    // fp8 W8A16: -, R, -, X, -, G, -, A, B, C, D, F
    {6.65, 1.09, 0, 0.241, 0.0725,
     {{}, {{1.0994, 1.2560, 1.5931}, 0}, {}, {{3.0932, 0, 0}, 2.89}, {}, {{1.9275, 0, 0}, 0.96}, {}, {{1.4369, 1.6295, 0}, 1.28},
      {{1.0004, 2.1533, 0}, 0}, {{1.3506, 1.5386, 2.0}, 0.09}, {{1.4295, 1.6564, 0}, 0.89}, {{1.7632, 3.5806, 0}, 1.43}}},
    // W8A8 (without the quantizer's launch): S, R, W, X, -, -, H, A, B, C, D, -
    {5.25, 2.58, 1.64, 0.200, 0.0018,
     {{{0.7889, 1.0025, 0}, 3.07}, {{0.5777, 0.7136, 0.9246}, 2.50}, {{1.2907, 0, 0}, 4.77}, {{1.6584, 0, 0}, 5.12}, {}, {},
      {{1.0419, 0, 0}, 4.78}, {{0.7811, 1.0186, 0}, 3.32}, {{0.7656, 1.5312, 0}, 4.77}, {{0.6406, 0.8521, 0}, 2.10},
      {{0.7151, 0.9370, 0}, 2.74}, {}}}};

// Partial sums of a call's K split: with the counters, within plm_gemm_noalloc's fixed scratch, so that it
// gives plm_gemm's bits. W8A8, which has no such form, may fill what its calls must bring anyway (K 17536,
// N 3344, M = 1130: 135 us whole, 99 with K in 2 and 31 MiB of sums). A tail's K split is bounded by the caller's bytes.
constexpr int64_t kMfmaMaxPartials = 24 << 20;

int64_t mfma_contract_bytes(plm_format f, int64_t m, int64_t n, int64_t k, bool a8);

mfma_config choose_mfma(plm_format f, int64_t m, int64_t n, int64_t k, bool a8, int64_t limit) {
    const mfma_mode mode = a8 ? kModeA8 : (f == PLM_FP8 ? kModeFp8 : kModeInt4);
    const mode_cost& mc = kModeCost[mode];
    const tuning& t = knobs();
    const int64_t cus = cu_count(), strips = ceil_div(n, kTileN), ktiles = ceil_div(k, kTileK);
    mfma_config best;
    double least = 0;
    const int64_t most = std::max(kCounterBytes + kMfmaMaxPartials, a8 ? mfma_contract_bytes(f, m, n, k, a8) : 0);
    int forced = -1;  // PLM_MFMA (tuning sweeps)
    for (int id = 0; id < kShapes; ++id)
        if (t.mfma_shape == kShapeLetter[id] && (kModeShapes[mode] >> id & 1)) forced = id;
    for (int id = 0; id < kShapes; ++id) {
        if (!(kModeShapes[mode] >> id & 1) || (forced >= 0 && id != forced)) continue;
        const shape sh = kShapeOf[id];
        const shape_cost& sc = mc.shapes[id];
        const int64_t m_blocks = ceil_div(m, sh.bm()), n_blocks = ceil_div(strips, sh.bs()), tiles = m_blocks * n_blocks;
        const double tile_mib = sh.bm() * sh.bs() * kTileN * 4.0 / (1 << 20);
        // us to bring in `of` tiles of the call's K: x rows and strips.
        auto memory = [&](int64_t of, int rows) {
            return static_cast<double>(of * ktiles) * (rows * (a8 ? 128 : 256) + sh.bs() * tile_bytes(f)) / 1e6 * mc.memory;
        };
        // `wgs` workgroups of tps K tiles over the CUs, no faster than `floor`.
        auto loop = [&](const shape_cost& sc, int64_t wgs, double tps, double floor) {
            const int slots = sc.step[2] > 0 ? 3 : (sc.step[1] > 0 ? 2 : 1);
            const double per_cu = wgs <= 4 * cus ? static_cast<double>(ceil_div(wgs, cus))
                                                 : static_cast<double>(wgs) / static_cast<double>(cus) + 0.5;
            const int whole = static_cast<int>(per_cu / slots);
            const double rest = per_cu - whole * slots;
            const int lo = static_cast<int>(rest);
            double g = whole * sc.step[slots - 1];
            if (rest > 0) g += lo + 1 > slots ? 0.0 : (lo > 0 ? sc.step[lo - 1] : 0.0) + (rest - lo) * (sc.step[lo] - (lo > 0 ? sc.step[lo - 1] : 0.0));
            const double steps = (tps + sc.fill) * g, x = steps * steps * steps, y = floor * floor * floor;
            return std::cbrt(std::sqrt(x * x + y * y));  // the larger one, rounded where they meet
        };
        auto exchange = [&](int64_t of, int64_t splits) {  // of `of` tiles' partial sums
            return mc.reduce + mc.reduce_pass * static_cast<double>(ceil_div(splits, split_batch(sh.mt, sh.ns)) - 1) +
                   mc.reduce_mib * tile_mib * static_cast<double>(of * splits);
        };
        for (int64_t want = 1; want <= std::min<int64_t>(8, ktiles); ++want) {
            const int64_t tps = ceil_div(ktiles, want), splits = ceil_div(ktiles, tps);
            if (splits != want || (t.mfma_splits > 0 && splits != std::min<int64_t>(t.mfma_splits, ktiles))) continue;
            if (splits > 1 && (t.mfma_unsplit || tiles > kMaxCounters || tiles * (splits - 1) >= 3 * cus || tps < 2)) break;
            mfma_config c;
            c.shape = id;
            c.m_blocks = static_cast<int>(m_blocks), c.n_blocks = static_cast<int>(n_blocks);
            c.splits = static_cast<int>(splits), c.tiles_per_split = static_cast<int>(tps);
            double cost = mc.launch + loop(sc, tiles * splits, static_cast<double>(tps), memory(tiles, sh.bm()));
            if (splits > 1) {
                const int64_t partials = tiles * splits * sh.bm() * sh.bs() * kTileN * 4;
                c.need = kCounterBytes + partials;
                if (c.need > most || c.need > limit) break;
                cost += exchange(tiles, splits);
            }
            // A tail launch: whole rounds, then the rest as halves or with K split, for the shapes of one workgroup
            // to a CU (beside others the first workgroups that end make room for the last ones; W8A8 H: 9 of
            // 10 sizes 5-30 % slower). Each launch brings in its own share of the tiles, and a tail's steps
            // take longer than a whole call's: 1.15 times for halves; 1.1 times for a K split, and 4 us and 6 us for
            // each MiB that the last workgroup adds up. The pick is then 0.2-0.8 % slower than the faster side, at
            // about 550 sizes where a tail can be had and comes near; 0.6-5.5 % without tails. us without and with
            // it: fp8 K 5120, N 34816, M = 2048 762, 676 (X); K 17408, N 5120, M = 2048 475, 370 (G); K 5120 138, 125;
            // int4 K 13696, N 3744, M = 2228 259, 230 (H); W8A8 K 16896, N 17440, M = 1007 409, 333 (W).
            const bool tails = sc.step[1] == 0 && !(mode == kModeA8 && id == kIdH);
            const int64_t rem = tiles % cus;
            if (tails && splits == 1 && tiles > cus && rem > 0 && 2 * rem <= cus && ktiles >= 8 && !t.mfma_no_tail &&
                !t.mfma_unsplit && t.mfma_splits == 0) {
                const double whole = mc.launch + loop(sc, tiles - rem, static_cast<double>(tps), memory(tiles - rem, sh.bm()));
                if (id == kIdX && mode != kModeFp8 && rem % m_blocks == 0 && !t.mfma_no_halves) {
                    // (fp8 W8A16, whose tall shape keeps the weights in registers, measured slower with halves.)
                    const double both = whole + 1.15 * loop(mc.shapes[kIdH], cus, static_cast<double>(tps), memory(2 * rem, kTallHalf.bm()));
                    if (both < cost) {
                        cost = both;
                        c.tail_tiles = static_cast<int>(rem), c.tail_halves = true;
                        c.tail_splits = 1, c.tail_tiles_per_split = static_cast<int>(ktiles);
                    }
                } else {
                    const int64_t ts = std::min<int64_t>(std::min<int64_t>(cus / rem, ktiles / 4), 8);
                    const int64_t ttps = ceil_div(ktiles, std::max<int64_t>(ts, 1)), tsp = ceil_div(ktiles, ttps);
                    const int64_t partials = rem * tsp * sh.bm() * sh.bs() * kTileN * 4;
                    const double steps = loop(sc, cus, static_cast<double>(ttps), memory(rem, sh.bm()));
                    const double both = whole + 1.1 * (steps + exchange(rem, tsp)) + 4.0 + 6.0 * tile_mib * static_cast<double>(tsp);
                    if (tsp >= 2 && rem <= kMaxCounters && kCounterBytes + partials <= limit && both < cost) {
                        cost = both;
                        c.tail_tiles = static_cast<int>(rem);
                        c.tail_splits = static_cast<int>(tsp), c.tail_tiles_per_split = static_cast<int>(ttps);
                        c.need = kCounterBytes + partials;
                    }
                }
            }
            if (best.shape < 0 || cost < least) least = cost, best = c;
        }
    }
    if (best.shape < 0) {  // a forced split that the shape or the workspace does not allow
        const shape sh = kShapeOf[kIdR];
        best.shape = kIdR;
        best.m_blocks = static_cast<int>(ceil_div(m, sh.bm())), best.n_blocks = static_cast<int>(ceil_div(strips, sh.bs()));
        best.tiles_per_split = static_cast<int>(ktiles);
    }
    return best;
}

// Workspace bytes a call must bring: a fixed contract (what callers size and what
// plm_gemm_noalloc refuses), which the plan above keeps within: a plan that would need more than
// the caller's workspace is not chosen. Each shape's K split fills the CUs once (a call with
// fewer tiles than CUs) or splits the tiles past whole rounds; the shape is the one with the
// fewest whole rounds of K tiles, weighted by the tile area over the shape's rate.
int64_t mfma_contract_bytes(plm_format f, int64_t m, int64_t n, int64_t k, bool a8) {
    struct old_shape {
        int bm, bs;
        double rate;
        bool ok;
    };
    const bool int4 = f == PLM_INT4, w8a16 = f == PLM_FP8 && !a8;
    // 128 x 128; 256 x 128; 256 x 256; 64 x 128; 256 x 192; 256 x 256 tall; the same by 8 wavefronts
    const old_shape shapes[9] = {{128, 8, w8a16 ? 0.5 : 0.75, true}, {256, 8, 0.7, true}, {256, 16, 1.0, !w8a16},
                                 {64, 8, 0.65, true}, {256, 12, 0.95, !w8a16}, {256, 16, w8a16 ? 0.75 : 1.03, true},
                                 {128, 8, 0.8, int4}, {64, 8, 0.7, int4}, {256, 8, 0.72, w8a16}};
    const int64_t cus = cu_count(), strips = ceil_div(n, kTileN), ktiles = ceil_div(k, kTileK);
    double least = 0;
    int64_t bytes = 0;
    for (int id = 0; id < 9; ++id) {
        const old_shape& sh = shapes[id];
        if (!sh.ok) continue;
        const int64_t m_blocks = ceil_div(m, sh.bm), tiles = m_blocks * ceil_div(strips, sh.bs), rem = tiles % cus;
        const double area = static_cast<double>(sh.bm) * sh.bs / sh.rate;
        const int64_t tile_bytes = int64_t{sh.bm} * sh.bs * kTileN * 4;
        int64_t want = 1;
        if (tiles < cus && tiles <= kMaxCounters) want = std::max<int64_t>(1, std::min<int64_t>(ceil_div(cus, tiles), ktiles / 4));
        const int64_t tps = ceil_div(ktiles, want), splits = ceil_div(ktiles, tps);
        double cost = static_cast<double>(ceil_div(tiles * splits, cus)) * (tps + 3 + (splits > 1 ? 0.5 * splits : 0.0)) * area;
        int64_t need = splits > 1 ? kCounterBytes + tiles * splits * tile_bytes : 0;
        if (splits == 1 && tiles > cus && rem > 0 && 2 * rem <= cus && rem <= kMaxCounters && ktiles >= 8) {
            const int64_t ts = std::min<int64_t>(cus / rem, ktiles / 4), ttps = ceil_div(ktiles, ts), tsp = ceil_div(ktiles, ttps);
            const int64_t full = (tiles - rem) / cus;
            if (id == 5 && !w8a16 && rem % m_blocks == 0) {
                cost = (static_cast<double>(full) * (tps + 3) + 0.55 * (ktiles + 3)) * area;
                need = 0;
            } else if (tsp >= 2) {
                cost = (static_cast<double>(full) * (tps + 3) + ttps + 3 + 0.5 * tsp) * area;
                need = kCounterBytes + rem * tsp * tile_bytes;
            }
        }
        if (id == 0 || cost < least) least = cost, bytes = need;
    }
    return bytes;
}

namespace {
// The plan within `limit` workspace bytes, and with any.
mfma_config plan_mfma(plm_format f, int64_t m, int64_t n, int64_t k, bool a8, int64_t limit = INT64_MAX) {
    thread_local plan_cache<mfma_config> cache;
    return cache.get(f + (a8 ? 2 : 0), m, n, k, limit, [&] { return choose_mfma(f, m, n, k, a8, limit); });
}
}  // namespace

int64_t mfma_contract(plm_format f, int64_t m, int64_t n, int64_t k, bool a8) {
    thread_local plan_cache<int64_t> cache;
    return cache.get(f + (a8 ? 2 : 0), m, n, k, 0, [&] { return mfma_contract_bytes(f, m, n, k, a8); });
}

int64_t mfma_workspace_bytes(plm_format f, int64_t m, int64_t n, int64_t k, bool a8) {
    return std::max(mfma_contract(f, m, n, k, a8), plan_mfma(f, m, n, k, a8).need);
}

namespace {
// Row blocks of an XCD's patch of work tiles. In id order with the row block fastest, an XCD gets the
// row blocks congruent to its number: with 8 of them one, and every XCD reads all of the weights
// through its fabric port; with 16 or 32 two or four, which is as good as a patch. Four rows cost the
// fewest bytes per XCD or nearly for every tile (1, 2, 8 and 16 measured too). id order -> patches of
// four: W8A8 K 17408, N 5120, M = 333 71 -> 64 us, M = 2048 214 -> 206; int4 K 4096, N 24576,
// M = 3300 527 -> 505, M = 4096 616 -> 620 (16 row blocks: left in id order).
int xcd_rows(int m_blocks) { return m_blocks % 16 == 0 ? 0 : std::min(4, m_blocks); }

void launch_mode(plm_format f, bool bf16, const mfma_args& a, int id, bool uniform, bool a8, dim3 grid, hipStream_t s) {
    if (a8) launch_plain_a8(a, bf16, id, grid, s);
    else if (f == PLM_INT4) launch_plain_int4(a, bf16, uniform, id, grid, s);
    else launch_plain_fp8(a, bf16, uniform, id, grid, s);
}
}  // namespace

int launch_mfma(const char* op, plm_format f, const void* x, bool bf16, const void* w, const void* scale,
                plm_dtype scale_dtype, int64_t m, int64_t n, int64_t k, int64_t block_n, int64_t group_size, void* y,
                void* workspace, size_t workspace_bytes, hipStream_t s, const uint8_t* xq, const float* x_scale) {
    PLM_CHECK_ARG(k <= (int64_t{1} << 21), op, "K above 2^21 is not supported");
    const bool a8 = xq != nullptr;
    const int64_t need = mfma_contract(f, m, n, k, a8);
    if (need > 0 && (workspace == nullptr || static_cast<int64_t>(workspace_bytes) < need)) {
        set_error(op, "workspace of %lld bytes required, %zu given", static_cast<long long>(need), workspace_bytes);
        return PLM_ERR_WORKSPACE;
    }
    const int64_t have = workspace != nullptr ? static_cast<int64_t>(workspace_bytes) : 0;
    mfma_config c = plan_mfma(f, m, n, k, a8);
    if (c.need > have) c = plan_mfma(f, m, n, k, a8, have);
    mfma_args a{};
    fill_common(a, x, w, scale, scale_dtype, m, n, k, block_n, group_size, y);
    a.splits = c.splits;
    a.tiles_per_split = c.tiles_per_split;
    a.m_blocks = c.m_blocks;
    a.n_blocks = c.n_blocks;
    a.xq = xq;
    a.x_scale = x_scale;
    if (c.need > 0) {
        a.counters = static_cast<uint32_t*>(workspace);
        a.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + kCounterBytes);
    }
    const bool uniform = group_size % kTileK == 0;
    const int tiles = c.m_blocks * c.n_blocks;
    if (c.tail_halves) {
        // Whole rounds of tall tiles, then the tail's columns of tiles as 128-row halves.
        const int nb_full = (tiles - c.tail_tiles) / c.m_blocks;
        a.n_blocks = nb_full;
        a.xcd_rows = xcd_rows(c.m_blocks);
        launch_mode(f, bf16, a, c.shape, uniform, a8, dim3(tiles - c.tail_tiles, 1), s);
        PLM_HIP_LAUNCH_CHECK(op);
        const int mb2 = static_cast<int>(ceil_div(m, kTallHalf.bm()));
        a.m_blocks = mb2;
        a.n_blocks = c.n_blocks;
        a.xcd_rows = 0;
        a.tile_base = nb_full * mb2;
        launch_mode(f, bf16, a, kIdH, uniform, a8, dim3((c.n_blocks - nb_full) * mb2, 1), s);
        PLM_HIP_LAUNCH_CHECK(op);
        return PLM_OK;
    }
    if (c.tail_tiles > 0) {
        // Whole rounds of unsplit tiles, then the tail tiles with K split.
        launch_mode(f, bf16, a, c.shape, uniform, a8, dim3(tiles - c.tail_tiles, 1), s);
        PLM_HIP_LAUNCH_CHECK(op);
        a.tile_base = tiles - c.tail_tiles;
        a.splits = c.tail_splits;
        a.tiles_per_split = c.tail_tiles_per_split;
        launch_mode(f, bf16, a, c.shape, uniform, a8, dim3(c.tail_tiles, c.tail_splits), s);
        PLM_HIP_LAUNCH_CHECK(op);
        return PLM_OK;
    }
    a.xcd_rows = xcd_rows(c.m_blocks);
    launch_mode(f, bf16, a, c.shape, uniform, a8, dim3(tiles, c.splits), s);
    PLM_HIP_LAUNCH_CHECK(op);
    return PLM_OK;
}

}  // namespace plm

extern "C" {
// Not part of the public ABI (include/pulsarlm_amd.h): the MFMA kernel's plan for a plain GEMM,
// for bench.py's report of the split-K / tail decomposition. out[0..7]: tile rows, tile
// columns, work tiles, K splits, tail tiles, tail K splits, tail as 128-row halves (0/1), and
// whether this build skips the split-K reduction (a measurement build, results invalid).
__attribute__((visibility("default"))) void plm_internal_mfma_plan(int format, int64_t m, int64_t n, int64_t k, int a8,
                                                                  int32_t* out) {
    using namespace plm;
    const mfma_config c = choose_mfma(static_cast<plm_format>(format), m, n, k, a8 != 0, INT64_MAX);
    const shape sh = kShapeOf[c.shape];
    out[0] = sh.bm();
    out[1] = sh.bs() * kTileN;
    out[2] = c.m_blocks * c.n_blocks;
    out[3] = c.splits;
    out[4] = c.tail_tiles;
    out[5] = c.tail_halves ? 1 : c.tail_splits;
    out[6] = c.tail_halves ? 1 : 0;
    out[7] = PLM_MEASURE_SKIP_REDUCTION;
}
}  // extern "C"
