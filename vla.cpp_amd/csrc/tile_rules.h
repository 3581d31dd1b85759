// Routing rules on sizes alone: which tile a launch takes.  Plain C++ without a device, so that a rule can be
// checked over its whole range on any host.
#pragma once

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
// kernel.  Two workgroups of 16 x 16 share a CU; beyond one round of them (512), 64-row tiles read the weights a quarter as
// often while they cover 33 to 64 rows (50 x 4096 x 720 gated 11.4 -> 9.3 us, 51 x 8192 x 1024 22.1 -> 18.9), and 16 x 16 tiles stay ahead
// of the tiled kernel up to four rounds: 200 x 1600 x 720 14.0 us, tiled 19.0; 482 x 640 x 960 14.9, 22.6; 100 x 4096 x 720 gated (1792
// workgroups) 18.9, 19.8; 150 x 4096 x 720 gated (2560) 23.4, 20.0.
inline int narrow_plan_f32(int M, int N) {
    const long wgs = narrow_wgs(M, N, 0);
    if (wgs <= 512) return 0;
    if (M <= 64) return M > 32 || wgs > 2048 ? 2 : 0;
    return wgs <= 2048 ? 0 : -1;
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

}  // namespace vla_rules
