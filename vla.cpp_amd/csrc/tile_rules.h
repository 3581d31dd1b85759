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

}  // namespace vla_rules
