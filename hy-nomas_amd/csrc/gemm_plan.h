// Which kernels an FP8 GEMM launch takes, by its shape alone: host code shared
// by the launcher and by the CPU test that pins the route of every GPU test's
// shape (tests/test_gemm_plan.py).
#pragma once
#include <algorithm>
#include <cmath>
#include <iterator>

#include "gemm_dma.h"

namespace hn {
namespace gemm {

constexpr int BM = 256, BN = 256, BK = 128;
enum Mode { ROWCOL = 0, BLOCKWISE = 1 };

constexpr int O_MIN_KT = 7;  // fewest K steps of the persistent kernel (its overlapped epilogue's passes + 3)

// The tail stripe (gemm_tail_kernel, tail_wide).
constexpr int TAIL_ROWS = 64;
constexpr int TAIL_COLS = 32;
constexpr int TAIL_WIDE_COLS = 384;
// Where the fused stripe gains (same-box A/B against the separate launch, two
// runs): the north star (32 light workgroups, K 3072) 0.978x and 0.981x, QKV
// (24, N 9216) 0.989x and 0.986x. Where it does not: past K 4096 an item
// outlasts the light workgroups' idle round (fc2, K 12 288: 1.013x), and with
// 8 light workgroups (out-projection, N 3072) it measured 0.991x and 1.017x.
constexpr int64_t TAIL_WIDE_MAX_K = 4096;
constexpr int TAIL_WIDE_MIN_LIGHT = 16;

// The tile of a launch, by an estimate of each shape's time in us:
//     3 + rounds * (g + K steps * c),
// with rounds the number of tiles per CU, rounded up (64 x 64 tiles run two to
// a CU: 0.3 more instead), and g (a tile's prologue and epilogue) and c (a
// K step) between their values for a few tiles and for a tile on every CU,
// where the loads from the L2s (11-15 TB/s in all) and the output's writes
// bound them. Fitted to back-to-back calls at K 512 to 12288 and 32 to 4608
// tiles; within 15 % of them, except where the weight comes from HBM. Below that
// range (K 128 to 384) the row/column pick is the fastest of the six in 19 of 21
// shapes of 65 to 4000 rows and 384 to 3072 columns, and 14 and 17 % off it in the
// two that give 256 x 192 tiles to every CU.
struct TileCost {
    int tm, tn;
    float g_low, c_low, g_full, c_full;
};

inline double tile_time(const TileCost& t, int64_t M, int64_t N, int64_t K, int cus, double g_min = 0.0) {
    const double tiles = (double)((M + t.tm - 1) / t.tm) * (double)((N + t.tn - 1) / t.tn);
    const double fill = std::min(1.0, tiles / cus);
    const double rounds = t.tm * t.tn <= 64 * 64 && tiles > cus ? tiles / cus + 0.3 : std::ceil(tiles / cus);
    const double g = std::max(g_min, t.g_low + (t.g_full - t.g_low) * fill), c = t.c_low + (t.c_full - t.c_low) * fill;
    return 3.0 + rounds * (g + (double)(K / BK) * c);
}

// gemm_small_kernel's shapes, per mode.
constexpr TileCost kSmallRowcol[] = {
    {64, 64, 1.3f, 0.18f, 1.3f, 0.18f},   {64, 128, 1.2f, 0.27f, 2.0f, 0.38f},
    {128, 128, 2.5f, 0.34f, 2.5f, 0.60f}, {128, 192, 2.5f, 0.43f, 3.0f, 0.75f},
    {128, 256, 2.0f, 0.57f, 4.5f, 0.86f}, {256, 192, 0.5f, 0.90f, 7.2f, 1.08f}};
constexpr TileCost kSmallBlockwise[] = {
    {64, 64, 1.0f, 0.25f, 1.0f, 0.25f}, {128, 128, 1.0f, 0.48f, 1.0f, 0.62f}, {128, 256, 1.4f, 0.75f, 2.0f, 1.02f}};
// The 256 x 256 tiles of gemm_rowcol_oe_kernel (its prologues and epilogues
// run beside other tiles' K steps, all but kBigOnce of them) and gemm_bw8_kernel.
constexpr TileCost kBigRowcol = {256, 256, 0.0f, 1.12f, 0.0f, 1.52f};
constexpr TileCost kBigBlockwise = {256, 256, 1.0f, 1.20f, 0.0f, 1.72f};
constexpr double kBigOnce = 4.0;

// The index of the small tile that a launch takes, or -1 for the 256 x 256
// tiles. Below O_MIN_KT steps the persistent kernel cannot run. A last stripe
// of at most TAIL_ROWS rows costs the 256 x 256 tiles no round. Within 3 % of
// each other the 256 x 256 tiles win. No row/column tile's prologue is taken for
// shorter than 64 x 64's: the fitted 0.5 us of 256 x 192 for a few tiles, outside
// the fit at K 128, gave it launches of two workgroups (65 x 128 -> 384 5.3 us,
// with 64 x 64 tiles 3.0 us); the floor changes no pick from K 256 on.
constexpr double kPrologueRowcol = 1.3;
inline int small_plan(int mode, int64_t M, int64_t N, int64_t K, int cus) {
    const bool row = mode == ROWCOL;
    if (M <= TAIL_ROWS && K / BK >= (row ? O_MIN_KT : 4)) return -1;  // the tail kernel alone
    const TileCost* const t = row ? kSmallRowcol : kSmallBlockwise;
    const int count = row ? (int)std::size(kSmallRowcol) : (int)std::size(kSmallBlockwise);
    const double g_min = row ? kPrologueRowcol : 0.0;
    auto small_time = [&](int i) { return tile_time(t[i], M, N, K, cus, g_min); };
    int best = 0;
    for (int i = 1; i < count; ++i)
        if (small_time(i) < small_time(best)) best = i;
    if (row && K / BK < O_MIN_KT) return best;
    const int64_t tail = M % BM, Mb = tail <= TAIL_ROWS && M > tail ? M - tail : M;
    const double big = kBigOnce + tile_time(row ? kBigRowcol : kBigBlockwise, Mb, N, K, cus);
    return small_time(best) < 0.97 * big ? best : -1;
}

// A launch's route: small tile `small`, or (small < 0) rows [0, Mt) in 256 x 256
// tiles (`tiles`; gemm_rowcol_oe_kernel on 8 S workgroups, or gemm_bw8_kernel) and
// the tail stripe [Mt, M), if any, on the persistent launch's light workgroups
// (tail_cols columns each) or, with tail_cols 0, on gemm_tail_kernel.
struct Route {
    int small;
    int64_t Mt;
    TileCounts tiles;
    int S;
    int tail_cols;
    int tail_waves, tail_blocks;  // gemm_tail_kernel: K split over 2 or 4 waves, 1 or 2 row blocks
};

// wg_cap: workgroups per XCD of a persistent launch, at most (0: the XCD's CUs).
inline Route gemm_route(int mode, int64_t M, int64_t N, int64_t K, int cus, int wg_cap = 0) {
    Route r{};
    r.small = small_plan(mode, M, N, K, cus);
    if (r.small >= 0) return r;
    // A last row stripe of at most TAIL_ROWS rows goes to gemm_tail_kernel (or,
    // in persistent launches, possibly to the light workgroups), and the tiles
    // cover only the rows above it: always in persistent launches; in
    // blockwise ones (one tile per workgroup, one workgroup per CU) when that
    // saves a whole round of tiles (the decoder's gate and up projections,
    // 10 800 x 4096 -> 12 288: 2064 tiles, 9 rounds, against 2016, 8) and K
    // has at least 4 scale blocks (a K step for each of up to 4 waves).
    const int64_t m_tail = M % BM;
    bool stripe = false;
    if (m_tail > 0 && m_tail <= TAIL_ROWS) {
        if (mode == ROWCOL) {
            stripe = true;
        } else if (K / BK >= 4) {
            const int64_t tn = (N + BN - 1) / BN, all = (M + BM - 1) / BM * tn, whole = M / BM * tn;
            stripe = (all + cus - 1) / cus > (whole + cus - 1) / cus;
        }
    }
    r.Mt = stripe ? M - m_tail : M;
    r.tiles = tile_counts(r.Mt, N);
    const int per_xcd_cus = cus / 8 > 0 ? cus / 8 : 1;
    const int cap = wg_cap >= 1 && wg_cap < per_xcd_cus ? wg_cap : per_xcd_cus;
    r.S = r.tiles.per_xcd < cap ? r.tiles.per_xcd : cap;
    // K is split over 2 waves, or 4 when the stripe has fewer 32-column groups
    // than CUs.
    r.tail_waves = N / TAIL_COLS < cus ? 4 : 2;
    r.tail_blocks = m_tail > 32 ? 2 : 1;
    if (stripe && mode == ROWCOL && r.Mt > 0) {
        // The tail stripe rides on the light workgroups (tail_wide) when
        // every XCD has some, at least TAIL_WIDE_MIN_LIGHT in all, there
        // are no edge tiles, each light workgroup's share of the columns
        // fits one item and K is at most TAIL_WIDE_MAX_K; else it has a
        // launch of its own.
        bool every = false;
        const int nl = light_count(r.tiles, r.S, &every);
        const int64_t cols = nl > 0 ? (N / 32 + nl - 1) / nl * 32 : 0;
        if (r.tiles.tiles_part == 0 && every && nl >= TAIL_WIDE_MIN_LIGHT && cols <= TAIL_WIDE_COLS &&
            K <= TAIL_WIDE_MAX_K)
            r.tail_cols = (int)cols;
    }
    return r;
}

}  // namespace gemm
}  // namespace hn
