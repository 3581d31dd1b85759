// Routing rules on sizes alone: which tile a launch takes.  Plain C++ without a device, so that a rule can be
// checked over its whole range on any host.
#pragma once

#include <cmath>

namespace vla_rules {

// Row blocks (16 rows) and column tiles (16 columns) per workgroup of the narrow-tile projection kernel.
constexpr int NARROW_PLANS[4][2] = {{1, 1}, {2, 1}, {4, 1}, {4, 2}};

inline int narrow_row_groups(int M, int p) { return (M + 16 * NARROW_PLANS[p][0] - 1) / (16 * NARROW_PLANS[p][0]); }
inline int narrow_col_groups(int N, int p) { return ((N + 15) / 16 + NARROW_PLANS[p][1] - 1) / NARROW_PLANS[p][1]; }
inline long narrow_wgs(int M, int N, int p) { return (long)narrow_col_groups(N, p) * narrow_row_groups(M, p); }
// Launched workgroups: the column groups are dealt out over the eight XCDs, each with all of its row groups, so that
// the busiest XCD has an eighth of this.
inline long narrow_grid(int M, int N, int p) { return (long)((narrow_col_groups(N, p) + 7) / 8 * 8) * narrow_row_groups(M, p); }

// Row blocks and column tiles per workgroup of the narrow-tile kernel: the split with the least
// operand traffic per CU among those whose workgroups are all on the chip at once.  A column
// tile (weights, from memory) weighs 2.2 times a row block (activations, from the L2): the
// ratio under which the rule picks the fastest split on the models' shapes at batch 1.  Without
// such a split the tiled kernel is the faster one -- 98 rows through 4608 x 1536: 288 narrow
// workgroups 14.0 us, tiled 11.0; 147 rows through 1536 x 6144: 144 workgroups 17.0, tiled 23.0 --
// and -1 is returned.
inline int narrow_plan(int M, int N, int K, bool qkv) {
    int p = -1, best = 1 << 30;
    for (int i = 0; i < 4; ++i) {
        const int rb = NARROW_PLANS[i][0], nb = NARROW_PLANS[i][1];
        if (rb > 1 && (rb / 2) * 16 >= M) continue;  // a smaller block holds every row
        // The QKV epilogue of 64 x 32 tiles (rotation, scatter) outweighs what so short a K saves: 64 rows of 6144 x 64 with the
        // norm inside 5.0 us, tiled 4.4; from K = 256 on the two are level or this one is ahead.
        if (qkv && i == 3 && K < 256) continue;
        const int cost = 5 * rb + 11 * nb;
        // The 96 KiB ring of 64 x 32 tiles leaves a CU to one workgroup: the 33rd on an XCD waits for a whole round.  300 rows
        // through 1600 x 720 with the norm inside: 250 workgroups, 35 on the busiest XCD, 10.2 us; tiled 6.9.
        const long wgs = i == 3 ? narrow_grid(M, N, i) : narrow_wgs(M, N, i);
        if (wgs <= 256 && cost < best) {
            best = cost;
            p = i;
        }
    }
    // More columns than one round holds: still this kernel up to 32 rows, where several of its workgroups share a CU (16
    // rows through 12288 x 1024 7.8 us, tiled 10.4).  From 33 rows on one fills a CU: 50 rows through 16384 x 1024, gated,
    // 12.7 us, tiled 11.6.
    return p < 0 && M <= 32 ? (M <= 16 ? 0 : 1) : p;
}

// Rows per workgroup of the fp32 narrow-tile kernel, as an index of NARROW_PLANS (16 x 16 or 64 x 16), or -1 for the tiled
// kernel.  Two workgroups of 16 x 16 share a CU; beyond one round of them (512), 64-row tiles read the weights of gated products
// a quarter as often while they cover 33 to 64 rows (50 x 4096 x 720 10.8 -> 8.6 us, 51 x 8192 x 1024 21.2 -> 18.2).  Their sums are four
// times as long (errors of 1.5e-7 and 2.1e-7 of the norm for K of 1024 and 2048, 16 x 16 tiles 1.0e-7 and 1.2e-7): plain and QKV
// products stay with 16 x 16 tiles, which are as fast there (51 x 2560 x 1024 9.1 us, 64-row tiles 9.0; 51 x 2560 x 2048 13.9, 15.4).  16 x 16
// tiles are ahead of the tiled kernel up to four rounds: 200 x 1600 x 720 14.0 us, tiled 19.0; 482 x 640 x 960 14.9, 22.6; 100 x 4096 x 720
// gated (1792 workgroups) 18.9, 19.8; 150 x 4096 x 720 gated (2560) 23.4, 20.0.  Up to 64 rows any number of rounds, for the tiled
// kernel's sums are the longest (5.7e-7 for K = 1024): up to 32 rows 16 x 16 tiles there too, since 64-row tiles would multiply
// repeated rows (16 x 36864 x 720 28.7 us, 64-row tiles 60.8, tiled 44.8; 8 x 151936 x 1024 130, 285, 192; 17 x 20480 x 720 21.5, 33.0, 30.1;
// 32 x 24576 x 2048 60.6, 86.7, 77.3; 32 x 65536 x 960 92.9, 132.6, 76.0).
inline int narrow_plan_f32(int M, int N, bool gated) {
    const long wgs = narrow_wgs(M, N, 0);
    if (wgs <= 512 || M <= 32 || (M <= 64 && !gated)) return 0;
    if (M <= 64) return 2;
    return wgs <= 2048 ? 0 : -1;
}

// XCD grid xm x xn = 8 for a tile grid of m_wg x n_wg workgroup tiles of tile_cols columns:
// every L2 reads its N tiles' rows of W once and its M tiles' rows of A once per panel of pn N
// tiles.  One panel while an XCD's rows of W fit in half of its 4 MiB L2 beside
// the streaming A and C; else panels of about 2 MiB of W.  The split with the least total,
// counting the padding of the tile grid.  forced_pn: 0 = by size, > 0 = that many tiles per panel.
struct XcdGrid {
    int xm, xn, pn;
    long wgs;  // workgroups of an XCD
};
inline XcdGrid xcd_grid(int M, int N, int K, int m_wg, int n_wg, double w_bytes_per_elem, int tile_cols, double a_bytes_per_elem, int forced_pn) {
    const double bytes_a = (double)M * K * a_bytes_per_elem, bytes_w = (double)N * K * w_bytes_per_elem;
    const double tile_w = (double)tile_cols * K * w_bytes_per_elem, l2_panel = 2.0 * 1024 * 1024;
    double best = -1;
    XcdGrid g = {1, 8, 1, 0};
    for (int xm = 1; xm <= 8; xm *= 2) {
        const int xn = 8 / xm;
        const int cn = (n_wg + xn - 1) / xn, cm = (m_wg + xm - 1) / xm;
        int pn = cn;
        if (forced_pn > 0) pn = forced_pn < cn ? forced_pn : cn;
        else if (cn * tile_w > l2_panel && cm >= 4) pn = tile_w >= l2_panel ? 1 : (int)(l2_panel / tile_w);
        const int panels = (cn + pn - 1) / pn;
        const long wgs = (long)cm * cn;
        const double cost = (bytes_a * xn * panels + bytes_w * xm) * (double)(wgs * 8) / ((double)m_wg * n_wg);
        if (best < 0 || cost < best) {
            best = cost;
            g = {xm, xn, pn, wgs};
        }
    }
    return g;
}

// Tile of the direct-to-LDS bf16 kernel (VLA_GEMM_TILE codes): enough 128 x 128 tiles to occupy the chip: use them (half the
// LDS and L2 traffic per multiply); else 128 x 64 tiles if those fill it; else 64 x 64 tiles, with 256-byte K rows (half the
// barriers per K) while one workgroup per CU covers them.
inline int dl_tile(int M, int n_tiles) {
    const long m128 = (M + 127) / 128, m64 = (M + 63) / 64;
    const long wgs0 = m128 * ((n_tiles + 1) / 2), wgs2 = m128 * n_tiles, wgs4 = m64 * n_tiles, wgs5 = m128 * ((n_tiles + 2) / 3);
    int cfg = wgs0 >= 128 ? 0 : (wgs2 >= 150 ? 2 : (wgs4 <= 256 ? 1 : 4));
    // 128x128 tiles that leave more than a third of the CUs idle lose to 128x64 tiles
    // that cover the chip in little more than one round (pi0's fused QKV: 140 -> 280)
    if (cfg == 0 && wgs0 < 160 && wgs2 <= 288) cfg = 2;
    // Between one and one and a half rounds of 128x128 tiles, some CUs would run two
    // workgroups while the rest run one; 128x192 tiles cover the same grid in a single
    // round of 1.5x workgroups (GR00T's fused QKV: 324 -> 216 workgroups).
    if (cfg == 0 && wgs0 > 256 && wgs0 <= 384 && wgs5 <= 256) cfg = 5;
    return cfg;
}

// Tile of an fp32 projection (VLA_GEMM_TILE codes): the fp32 MFMA is its whole time, a 128 x 64 tile takes 1.6 times as long
// as a 64 x 64 one and a 128 x 128 one three times, and further rounds of workgroups cost somewhat less than the first because
// two share a CU.  A grid just past a round is what the bf16 rule got wrong here: 1323 x 1536 x 1536 on 264 of 128 x 64 110 us, on
// 504 of 64 x 64 63; 3549 x 704 x 960 75 and 57.  On 140 measured shapes (65 to 6500 rows, N 256 to 4096) 0.95 of the time of that
// rule's tiles (geometric mean), none more than 3 % slower; 3144 x 896 x 1536 stays level (112 us on each).
inline int f32_tile(int M, int n_tiles) {
    const long m128 = (M + 127) / 128, m64 = (M + 63) / 64;
    const long wgs0 = m128 * ((n_tiles + 1) / 2), wgs2 = m128 * n_tiles, wgs4 = m64 * n_tiles;
    auto rounds = [](long wgs, double more) {
        const long n = (wgs + 255) / 256;
        return n == 1 ? 1.0 : more * n;
    };
    const double t4 = rounds(wgs4, 0.72), t2 = 1.6 * rounds(wgs2, 0.9), t0 = 3.05 * rounds(wgs0, 0.9);
    if (t4 <= t2 && t4 <= t0) return wgs4 <= 256 ? 1 : 4;
    return t2 <= t0 ? 2 : 0;
}

// Predicted time (us) of a bf16 projection on a tile: `fixed`, and per round of workgroups on the busiest XCD (32 CUs) its
// prologue and epilogue `round` (QKV: + `qkv`, with a LayerNorm inside + `layer`) and `step` per 64 k, which grows by `load` with the
// share of the CUs that are busy.  Tiles of which two share a CU: round2 and step2 for the rounds of two.  Fitted to 3362
// measured shapes (200 to 16000 rows, N 256 to 10240, K 128 to 8192, plain, gated, QKV); the prediction is off by 11 % (rms).
struct TileTime {
    int rows, cols;
    bool pairs;
    double fixed, round, step, load, round2, step2, qkv, layer;
    double us(int M, int N, int K, int kind) const {
        const XcdGrid g = xcd_grid(M, N, K, (M + rows - 1) / rows, (N + cols - 1) / cols, 2.0, cols, 2.0, 0);
        const double w = g.wgs / 32.0, kt = (K + 63) / 64, extra = kind == 0 ? 0.0 : kind == 1 ? qkv : layer;
        const long n = (g.wgs + 31) / 32, n2 = pairs ? n / 2 : 0, n1 = n - 2 * n2;
        return fixed + n2 * (round2 + 1.5 * extra + kt * step2) + n1 * (round + extra + kt * (step + load * (w < 1 ? w : 1)));
    }
};

// Tile of the wide-tile kernel: rows x columns, and whether two workgroups share a CU.  PLAIN_*: plain epilogue only.
enum { WIDE_256X256 = 0, WIDE_192X192, WIDE_256X128, WIDE_192X128, WIDE_128X128, WIDE_128X128_PAIRS, WIDE_TILES,
       PLAIN_96X96_PAIRS = WIDE_TILES, PLAIN_128X96, PLAIN_96X64_PAIRS, PLAIN_TILES };

// The wide tile with the least predicted time, or -1 where the direct-to-LDS kernel's tile is not predicted 6 % slower.  kind:
// 0 plain or gated, 1 QKV, 2 QKV with a LayerNorm inside.  On the fitted shapes the wide tile is taken on 60 %, where it needs
// 0.84 of the time (geometric mean; 0.90 over all, 0.89 if the faster one were always known); 1 % of them are 3 to 7 %
// slower, one 15 % (576 x 2752 x 5552 gated, 71.6 -> 82.0 us).  1323 x 6144 x 1536 46.3 -> 28.3 us (192 x 192: 224 workgroups, one
// round, where 528 of 128 x 128 left 16 for a second one), 816 x 8192 x 1024 gated 21.4 -> 19.6, 13824 x 3072 x 2048 186 -> 144
// (256 x 256), 4096 x 4096 x 4096 147 -> 102 (weights not in the caches).
inline int wide_tile(int M, int N, int K, int kind, double* predicted = nullptr) {
    static const TileTime wide[WIDE_TILES] = {
        {256, 256, false, 0.18, 11.50, 1.234, 0.314, 0, 0, 1.57, 3.50}, {192, 192, false, 1.05, 7.02, 0.703, 0.225, 0, 0, 2.04, 3.15},
        {256, 128, false, 1.05, 6.86, 0.676, 0.188, 0, 0, 1.31, 2.89},  {192, 128, false, 1.38, 5.32, 0.565, 0.152, 0, 0, 1.51, 2.93},
        {128, 128, false, 1.85, 3.90, 0.455, 0.115, 0, 0, 1.10, 2.04},  {128, 128, true, 1.41, 2.86, 0.664, 0.198, 4.82, 0.982, 1.08, 1.63}};
    static const TileTime dl[6] = {
        {128, 128, true, 2.34, 4.32, 0.249, 0.410, 5.77, 1.132, -0.38, 0.29}, {64, 64, false, 2.23, 2.14, 0.194, 0.029, 0, 0, -0.16, 0.87},
        {128, 64, true, 3.53, 1.36, 0.335, 0.063, 2.32, 0.662, 0.13, 0.81},   {128, 64, true, 3.53, 1.36, 0.335, 0.063, 2.32, 0.662, 0.13, 0.81},
        {64, 64, true, 4.86, 1.00, 0.300, 0.300, 0.00, 0.378, -0.42, 0.31},   {128, 192, false, 6.38, 2.96, 0.637, 0.119, 0, 0, 0.21, 0.71}};
    const int cfg = dl_tile(M, (N + 63) / 64);
    const double dl_us = dl[cfg].us(M, N, K, kind);
    double least = 0.94 * dl_us;
    int best = -1;
    for (int t = 0; t < WIDE_TILES; ++t) {
        // one 128 x 128 tile per CU, where 128 x 64 tiles cover the chip: up to 18 % slower than those
        if (t == WIDE_128X128 && cfg != 0) continue;
        const double us = wide[t].us(M, N, K, kind);
        if (us < least) {
            least = us;
            best = t;
        }
    }
    if (predicted) *predicted = best < 0 ? dl_us : least;
    return best;
}

// The same for a plain product, whose epilogue also comes with 32- and 48-column wavefronts: one of those tiles where it is predicted 6 %
// faster than what wide_tile takes.  Their step per 64 k is the root of the squares of what a CU needs for itself and what its share of the
// L2s' rate allows (load, times the share of the CUs that are busy): 1323 x 1536 x 6144 takes 46.1 us on 224 tiles of 96 x 96, 42.6 on 176 of
// 128 x 96.  On 947 shapes (200 to 4000 rows, N 256 to 8192, K 128 to 8192, weights from memory) taken on 253, where it needs 0.88 of the time
// (geometric mean); five of them are up to 6 % slower.  Long rows that do not start on a cache line are left out: predicted as well on the mean,
// but 672 x 1536 x 4432 and 1042 x 1152 x 5008 take 1.22 times as long.  1323 x 1536 x 6144 55.2 -> 42.6 us, 2000 x 1536 x 6144 59.1 -> 48.4, 1600 x 720 x 2048
// 13.8 -> 12.0; 408 x 1536 x 6144 stays: 24.4, here 29.4.  Outside of those limits (16 to 20000 rows, N 8 to 40000, K 16 to 20000; 406 shapes for which it names a
// tile) it needs 0.89 of the time, at most 1.03, but for two k tiles of up to 32 columns, which stay: 6301 x 8 x 112 3.5 us, here 3.8; 7527 x 32 x 96 3.6, 3.9.
inline int plain_tile(int M, int N, int K) {
    static const struct { int rows, cols; bool pairs; double fixed, round, step, load, round2, step2; } t[PLAIN_TILES - WIDE_TILES] = {
        {96, 96, true, 1.08, 3.64, 0.357, 0.329, 4.44, 0.708}, {128, 96, false, 1.33, 4.80, 0.410, 0.285, 0, 0}, {96, 64, true, 1.94, 1.93, 0.287, 0.200, 2.31, 0.609}};
    double least;
    int best = wide_tile(M, N, K, 0, &least);
    if ((K % 64 != 0 && K > 1024) || (N <= 32 && K > 64 && K <= 128)) return best;
    least *= 0.94;
    for (int i = 0; i < PLAIN_TILES - WIDE_TILES; ++i) {
        const XcdGrid g = xcd_grid(M, N, K, (M + t[i].rows - 1) / t[i].rows, (N + t[i].cols - 1) / t[i].cols, 2.0, t[i].cols, 2.0, 0);
        const long n = (g.wgs + 31) / 32, n2 = t[i].pairs ? n / 2 : 0, n1 = n - 2 * n2;
        const double load = t[i].load * (g.wgs < 32 ? g.wgs / 32.0 : 1.0), kt = (K + 63) / 64;
        const double us = t[i].fixed + n2 * (t[i].round2 + kt * t[i].step2) + n1 * (t[i].round + kt * std::sqrt(t[i].step * t[i].step + load * load));
        if (us < least) {
            least = us;
            best = WIDE_TILES + i;
        }
    }
    return best;
}

// Tile of a ternary GEMM (VLA_TERNARY_TILE codes) by predicted time: a launch costs `fixed`, and
// `step` per 128 k while every workgroup has a CU of its own; up to two workgroups per CU
// overlap to `two` steps, beyond that a step takes `more` times the workgroups per CU.  The
// constants (us) are a fit to 75 measured shapes (40 to 4096 rows; N 640, 2560, 3840, 13824; K
// 2560, 6912).  On 234 shapes (33 to 4664 rows; N 256 to 32000; K 512 to 16384) the picked tile is within
// 4 % of the fastest of the six on 227 and within 11 % on all.  The prediction's error is a few per cent, so
// that 128 x 256 tiles, where they fill half the chip, give way only to a tile predicted 4 % faster: 2048 x
// 2560 x 6912 45.4 -> 44.0 us, 2048 x 3840 x 2560 22.6 -> 21.9 (64 x 128 and 64 x 256 tiles without the margin).
inline int ternary_tile(long M, long N, long K) {
    const struct { int tile, rows, cols; double fixed, step, two, more; } t[] = {
        {21, 32, 64, 3.23, 0.170, 1.48, 0.88},   {19, 64, 64, 3.35, 0.224, 1.32, 1.04},   {18, 64, 128, 4.55, 0.311, 1.56, 1.00},
        {17, 128, 128, 6.09, 0.490, 1.65, 1.04}, {20, 64, 256, 5.30, 0.546, 1.53, 0.97}, {16, 128, 256, 6.79, 0.762, 1.36, 1.13}};
    int best = 16;
    double least = 1e30;
    for (const auto& x : t) {
        const double r = (double)(((M + x.rows - 1) / x.rows) * ((N + x.cols - 1) / x.cols)) / 256.0;
        const double us = x.fixed + K / 128 * x.step * (r <= 1 ? 1.0 : r <= 2 ? x.two : (x.more * r > x.two ? x.more * r : x.two));
        const double margin = x.tile == 16 && r >= 0.5 ? 0.96 : 1.0;
        if (us * margin < least) {
            least = us * margin;
            best = x.tile;
        }
    }
    return best;
}

// Whether a bf16 attention launch of 48- or 64-wide heads (`grid` workgroups of 32 rows, `blocks` 64-key tiles) takes a wavefront
// per tile (attn_tiles_kernel, the bits of the tiled kernel) instead of the tiled kernel, which reads K and V^T once per 64
// to 128 rows but walks the keys.  Two rounds of workgroups while a CU holds two of them, else one: 50 rows x 15 heads on 5, 227
// keys: 1, 4, 8, 16, 20 observations (40, 120, 200, 400, 520 workgroups) 7.9, 8.2, 8.2, 8.4, 9.6 us tiled and 5.5, 5.7, 5.8, 6.9, 9.8
// here; 291 keys (five tiles) 1, 4, 9, 10 observations (40, 120, 240, 280) 9.2, 9.4, 9.6, 9.5 and 6.0, 6.2, 6.4, 10.0; 512 keys 1 and 9
// observations 9.5, 9.9 and 6.6, 7.1; 48-wide, 49 rows, 32 heads: 227 keys 1, 4, 8 observations (64, 256, 512) 6.9, 7.1, 7.2 and 5.1, 5.4, 6.3.
constexpr int ATTN_TILES_MAX = 10;  // tiles that a workgroup's LDS holds
inline bool attn_tiles(long grid, int blocks) {
    return grid <= (blocks <= 4 ? 512 : 256);
}

// Whether an fp32 attention launch of 48- or 64-wide heads takes 16 rows per workgroup with the 32-key blocks shared out over
// its wavefronts (`grid` workgroups, `blocks` key blocks) instead of the tiled kernel.  About two rounds of workgroups: 50 rows x
// 15 heads on 5, 227 keys: 1, 4, 8, 16 observations (50, 200, 400, 800 workgroups) 13.0, 25.2, 25.9, 26.6 us tiled and 7.3, 7.8, 13.4, 23.9
// here; where the tiled kernel slices the keys over workgroups, more than two blocks per wavefront (ten of them) are left to
// it: 16 rows x 16 heads on 4, 1000 keys 14.8 us, here 16.0 (one slice only: 50 x 15 on 5, two observations 87.9, here 17.1).
inline bool attn_rows(long grid, int blocks, bool sliced) { return grid <= 512 && (blocks <= 20 || !sliced); }

// Whether a bf16 attention launch of 128-wide heads with three or four row tiles a workgroup takes the tiled kernel's direct-to-LDS form rather than
// the register-staged one: more workgroups than CUs, so that a CU has two.  515 rows of 20 heads on 5 kv heads, two-term probabilities: 3 observations
// (255 workgroups) 24.8 us, direct 28.4; 4, 8, 12 (340, 680, 1020) 42.9, 64.8, 86.2, direct 37.6, 59.1, 72.3; 16 of 100 rows 18.5, direct
// 14.8.  dl: the tuning override VLA_ATTN_DL, 0 pins the register-staged form.
inline bool attn_ring128(long wgs, bool aligned, int dl) { return dl != 0 && aligned && wgs > 256; }

// Row blocks (of 16) per workgroup and key slices of a bf16 attention launch of 256-wide heads on attn_wide_kernel, or rb = 0 for the tiled
// kernel.  pairs: (observation, kv head); units: 64-key units, four of which a workgroup walks at a time; part_rows: rows of partials
// that the call's scratch holds (what the tiled kernel asks for, so that no call needs more than it did).  A workgroup fills a CU, so only splits whose
// workgroups all run at once (32 on the busiest XCD) are taken: behind them the tiled kernel is the faster one, which reads K and
// V^T once per 128 rows (50 positions x 8 heads on 955 keys, 20 observations, 260 workgroups: tiled 40.5 us, here 41.7; 32: 34.6, 46.8).  Of
// these the least predicted time (us): start and end 5.5, a round of units 2.5 (16 rows) or 3.3 (32), the merge launch 1.8 and 0.75 per
// 1000 partial rows.  Against the tiled kernel and its merge, 50 positions, 955 keys from memory: 1, 2, 4, 8, 12, 16 observations 16.6, 18.3, 19.1,
// 22.0, 31.2, 27.8 us, here 10.8, 13.1, 15.6, 16.2, 21.2, 21.9; 60 to 330 keys at 1 to 16 observations 0.59 to 0.95 of its time.  Left to the
// tiled kernel (of 1067 launches of 8 to 800 rows on 60 to 3000 keys, 1 to 64 observations, 932 are taken, in 0.70 of its time (geometric mean, 1.06 at most)):
//  - 16 rows or fewer on 5 to 8 units, on up to 11 of up to four pairs; up to 32 rows on 5 to 8 of up to six: two rounds for what one wavefront row of the
//    tiled kernel's slices does as fast (8 rows, 281 keys 9.1 us, here 9.8; 8 rows, 523 keys 8.8, 9.8; 16 rows, 523 keys 9.6, 10.3);
//  - more than 5 MiB of K and V^T for an XCD's 4 MiB L2 and more than 32 rows: its row tiles start at different units, and what one has
//    read is gone before the next one comes (128 rows, 1990 keys: 32 pairs 31.1 us, here 72.7; 24 pairs 26.5, 36.9; 20 pairs 34.0, 27.1);
//  - more than 256 rows on more than 24 units of five to eight pairs: level on the mean, 0.79 to 1.20 of its time (400 rows, eight pairs, 3000 keys 27.1, 32.5).
struct WideHeads {
    int rb, slices;
};
inline WideHeads wide_heads(long pairs, int rows, int units, long part_rows, bool forced) {
    WideHeads best = {0, 1};
    if (!forced) {
        if (rows <= 16 ? units > 4 && (units <= 8 || (units <= 11 && pairs <= 4)) : rows <= 32 && units > 4 && units <= 8 && pairs <= 6) return best;
        if (rows > 32 && (pairs + 7) / 8 * units > 80) return best;  // a unit of a pair is 64 KiB
        if (rows > 256 && pairs > 4 && pairs <= 8 && units > 24) return best;
    }
    double least = 1e30;
    for (int rb = 1; rb <= 2; ++rb) {
        const long tiles = (rows + 16 * rb - 1) / (16 * rb);
        for (int s = 1; s <= 16 && s <= units; ++s) {
            const int per = (units + s - 1) / s;
            const long partials = s > 1 ? pairs * s * tiles * 16 * rb : 0, rounds = ((pairs * s + 7) / 8 * tiles + 31) / 32;
            if ((units + per - 1) / per != s || partials > part_rows || (rounds > 1 && !forced)) continue;  // (no empty slice)
            const double us = rounds * (2.9 + (per + 3) / 4 * (rb == 1 ? 2.5 : 3.3)) + 2.6 + (s > 1 ? 1.8 + 0.75e-3 * partials : 0.0);
            if (us < least) {
                least = us;
                best = {rb, s};
            }
        }
    }
    return best;
}

}  // namespace vla_rules
