"""The kernels' routing rules on sizes (csrc/tile_rules.h), over their whole range, on the host."""
import ctypes
import os
import subprocess

import pytest

from util import ROOT


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = str(d / "rules.cpp"), str(d / "rules.so")
    with open(src, "w") as f:
        f.write('''#include "tile_rules.h"
extern "C" int plan(int M, int N, int K, int qkv) { return vla_rules::narrow_plan(M, N, K, qkv); }
extern "C" int plan_f32(int M, int N, int gated) { return vla_rules::narrow_plan_f32(M, N, gated); }
extern "C" int rows_kernel(int grid, int blocks, int sliced) { return vla_rules::attn_rows(grid, blocks, sliced); }
extern "C" int tiles_kernel(int grid, int tiles) { return vla_rules::attn_tiles(grid, tiles); }
extern "C" int f32_tile(int M, int n_tiles) { return vla_rules::f32_tile(M, n_tiles); }
extern "C" int ring128(int wgs, int aligned, int dl) { return vla_rules::attn_ring128(wgs, aligned, dl); }
extern "C" int wide(int M, int N, int K, int kind) { return vla_rules::wide_tile(M, N, K, kind); }
extern "C" int plain(int M, int N, int K) { return vla_rules::plain_tile(M, N, K); }
extern "C" int ternary(int M, int N, int K) { return vla_rules::ternary_tile(M, N, K); }
extern "C" int heads256(int pairs, int rows, int units, int part_rows, int forced) {
    const vla_rules::WideHeads h = vla_rules::wide_heads(pairs, rows, units, part_rows, forced);
    return h.rb * 100 + h.slices;
}
extern "C" int rows(int p) { return 16 * vla_rules::NARROW_PLANS[p][0]; }
extern "C" int cols(int p) { return 16 * vla_rules::NARROW_PLANS[p][1]; }
''')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "vla.cpp_amd", "csrc"), src, "-o", so],
                   check=True)
    return ctypes.CDLL(so)


# 16-column steps up to the widest model, then wider
WIDTHS = list(range(16, 8449, 16)) + [12288, 16384, 32768, 151936]


def test_no_xcd_gets_more_narrow_tiles_of_64_x_32_than_it_has_cus(rules):
    """A CU holds one workgroup of that size (96 KiB of LDS each) and an XCD has 32 CUs; the column groups are
    dealt out over eight XCDs, each with all of its row groups."""
    taken = 0
    for M in range(65, 513):
        for N in WIDTHS:
            p = rules.plan(M, N, 720, 0)
            if p >= 0 and (rules.rows(p), rules.cols(p)) == (64, 32):
                taken += 1
                groups = -(-N // 32)
                assert -(-groups // 8) * -(-M // 64) <= 32, (M, N)
    assert taken > 10000


def test_narrow_tiles_of_more_columns_than_one_round_only_up_to_32_rows(rules):
    """Beyond, a workgroup of the 64-row tiles fills a CU and the columns would take several rounds."""
    for N in WIDTHS:
        if N > 8192:
            assert all(rules.plan(M, N, 720, 0) >= 0 for M in range(1, 33)), N
            assert all(rules.plan(M, N, 720, 0) < 0 for M in range(33, 513)), N


def test_short_fused_qkv_projections_stay_off_64_x_32_tiles(rules):
    """Below K = 256 the tiled kernel is the faster one there; smaller tiles, plain projections and K from
    256 on are not touched."""
    for M in range(33, 513, 7):
        for N in WIDTHS:
            long_k, short_k = rules.plan(M, N, 256, 1), rules.plan(M, N, 128, 1)
            assert long_k == rules.plan(M, N, 128, 0)
            assert short_k == (-1 if long_k == 3 else long_k), (M, N)


# M, N, K -> measured us on the tiles 16 (128 x 256), 17 (128 x 128), 18 (64 x 128), 19 (64 x 64), 20 (64 x 256), 21 (32 x 64)
TERNARY_US = [
    ((2048, 3840, 2560), (21.8, 22.1, 25.7, 32.1, 22.6, 37.0)),
    ((2048, 2560, 6912), (43.9, 44.0, 45.2, 46.8, 49.4, 58.2)),
    ((3000, 2560, 2560), (21.7, 22.3, 25.9, 32.1, 22.8, 37.3)),
    ((4096, 3840, 2560), (33.0, 41.0, 48.0, 58.7, 43.3, 69.6)),
    ((4664, 13824, 2560), (132.7, 159.4, 184.2, 234.8, 155.7, 275.2)),
    ((512, 2560, 2560), (20.8, 15.6, 10.8, 9.2, 16.2, 10.3)),
    ((583, 13824, 2560), (31.4, 32.9, 31.5, 36.4, 33.7, 41.2)),
    ((583, 2560, 6912), (42.7, 31.8, 22.2, 18.0, 34.3, 28.1)),
    ((1024, 3840, 2560), (21.0, 16.0, 14.3, 17.7, 16.7, 21.6)),
    ((64, 640, 2560), (20.4, 15.3, 10.5, 7.8, 16.1, 6.9)),
    ((300, 4096, 4096), (28.3, 21.0, 14.6, 11.9, 22.6, 13.7)),
    ((4096, 512, 512), (10.1, 8.0, 5.8, 5.2, 7.7, 6.3)),
    ((1500, 8192, 1024), (17.8, 19.4, 20.5, 26.7, 19.3, 31.4)),
]


@pytest.mark.parametrize("shape,us", TERNARY_US)
def test_ternary_tile_is_near_the_fastest_and_not_slower_than_the_large_tiles(rules, shape, us):
    """Within the prediction's error (4 %) of the fastest tile, and 128 x 256 tiles, where they fill half the
    chip, are left only for a faster one (2 %: two runs of one tile)."""
    M, N, K = shape
    took = us[rules.ternary(M, N, K) - 16]
    assert took <= 1.04 * min(us)
    if -(-M // 128) * -(-N // 256) >= 128:
        assert took <= 1.02 * us[0]


def test_fp32_narrow_tiles_of_more_than_one_round(rules):
    """16 x 16 tiles up to four rounds of two per CU and always a narrow tile for up to 64 rows; 64-row tiles only for gated products of
    33 to 64 rows beyond one round (elsewhere they repeat the weights, waste rows or make sums longer)."""
    for M in list(range(1, 130)) + [200, 300, 400, 512]:
        for N in WIDTHS:
            for gated in (0, 1):
                wgs, p = -(-M // 16) * (N // 16), rules.plan_f32(M, N, gated)
                want = -1 if M > 64 and wgs > 2048 else 2 if gated and 32 < M <= 64 and wgs > 512 else 0
                assert p == want, (M, N, gated)


# M, N, K, kind (0 plain or gated, 1 QKV, 2 with a LayerNorm) -> measured us of the direct-to-LDS kernel and on the wide tiles
# 256 x 256, 192 x 192, 256 x 128, 192 x 128, 128 x 128, 128 x 128 in pairs
WIDE_US = [
    ((1323, 6144, 1536, 0), 53.3, (45.2, 30.2, 47.2, 45.5, 47.1, 46.1)),
    ((816, 8192, 1024, 0), 22.3, (28.5, 20.7, 19.8, 28.6, 23.8, 20.0)),
    ((1600, 4096, 720, 0), 17.1, (22.9, 16.7, 16.6, 24.2, 20.5, 16.5)),
    ((408, 6144, 1536, 0), 21.1, (45.6, 25.1, 25.7, 21.3, 18.0, 26.0)),
    ((1323, 4608, 1536, 2), 34.8, (44.8, 30.9, 30.5, 45.0, 36.2, 30.8)),
    ((13824, 3072, 2048, 1), 202.2, (160.0, 163.7, 173.4, 177.5, 199.3, 175.9)),
    ((4096, 4096, 4096, 0), 149.3, (106.6, 166.1, 117.2, 144.6, 146.7, 138.5)),
    ((816, 1024, 4096, 0), 19.5, (85.8, 47.2, 44.6, 38.8, 32.4, 55.8)),
    ((816, 2560, 1024, 1), 11.3, (28.3, 19.2, 17.7, 15.9, 13.3, 15.3)),
    ((1088, 1536, 1536, 0), 12.1, (36.8, 22.4, 21.2, 18.2, 15.3, 19.1)),
    ((5300, 4864, 4576, 1), 332.9, (239.2, 237.4, 297.1, 287.4, 352.1, 337.8)),
    ((4886, 448, 288, 0), 8.7, (17.9, 12.0, 11.9, 10.0, 8.8, 8.3)),
    ((600, 1344, 336, 1), 5.2, (19.2, 13.8, 12.8, 11.4, 9.8, 9.4)),
    ((8362, 4160, 496, 0), 75.2, (73.7, 69.8, 73.3, 78.6, 87.2, 64.6)),
    ((3570, 8512, 1440, 0), 133.2, (141.7, 112.2, 118.2, 135.9, 142.3, 121.7)),
]


@pytest.mark.parametrize("shape,dl,wide", WIDE_US)
def test_wide_tiles_are_taken_where_they_are_faster(rules, shape, dl, wide):
    """The picked kernel is not slower than the direct-to-LDS one, and within the prediction's error (11 %) of the fastest."""
    t = rules.wide(*shape)
    took = dl if t < 0 else wide[t]
    assert took <= dl
    assert took <= 1.11 * min(wide + (dl,))


def test_a_wide_tile_is_named_for_every_size(rules):
    """From one row to millions the rule answers with a tile or none (no size divides by zero or overflows)."""
    for M in (1, 63, 64, 513, 1000, 65536, 1 << 24):
        for N in (8, 64, 200, 4096, 151936):
            for K in (16, 720, 8192, 1 << 20):
                for kind in (0, 1, 2):
                    assert -1 <= rules.wide(M, N, K, kind) < 6


def test_attention_rows_only_while_the_workgroups_are_few(rules):
    for blocks in (1, 8, 9, 20, 21, 1000):
        for sliced in (0, 1):
            assert rules.rows_kernel(512, blocks, sliced) == (blocks <= 20 or not sliced) and not rules.rows_kernel(513, blocks, sliced)
    for tiles in range(1, 11):
        assert rules.tiles_kernel(256, tiles) and not rules.tiles_kernel(513, tiles)
        assert rules.tiles_kernel(512, tiles) == (tiles <= 4)


# M, N, K -> measured us on the tiles 0 (128 x 128), 1 (64 x 64, 256-byte K rows), 2 (128 x 64), 4 (64 x 64)
F32_US = [((1323, 1536, 1536), (113.1, 65.2, 110.0, 62.8)), ((408, 1536, 1536), (111.2, 36.6, 63.1, 37.7)), ((1600, 720, 720), (57.7, 33.7, 33.8, 32.2)),
          ((816, 1024, 1024), (75.7, 26.0, 43.6, 26.2)), ((3549, 704, 960), (75.1, 59.7, 71.4, 57.2)), ((3144, 896, 1536), (113.7, 117.9, 108.8, 111.0)),
          ((964, 640, 960), (72.0, 23.7, 40.6, 25.0)), ((700, 1536, 1536), (111.1, 61.1, 62.9, 61.1))]


@pytest.mark.parametrize("shape,us", F32_US)
def test_fp32_tile_is_near_the_fastest(rules, shape, us):
    took = dict(zip((0, 1, 2, 4), us))[rules.f32_tile(shape[0], -(-shape[1] // 64))]
    assert took <= 1.04 * min(us)


def test_256_wide_heads_keep_to_their_scratch_and_to_one_round(rules):
    """A split fits the partial rows that the tiled kernel would have used, leaves no slice empty and no XCD more than 32
    workgroups; what does not fit one round is the tiled kernel's, unless forced."""
    taken = 0
    for pairs in list(range(1, 34)) + [64, 100, 1000]:
        for rows in (1, 8, 16, 17, 32, 33, 136, 400, 408, 800, 1600, 5000):
            for units in list(range(1, 40)) + [128, 1000]:
                for part_rows in (0, 512, 2560, 3584, 100000):
                    rb, s = divmod(rules.heads256(pairs, rows, units, part_rows, 0), 100)
                    assert divmod(rules.heads256(pairs, rows, units, part_rows, 1), 100)[0] in (1, 2)
                    if not rb:
                        continue
                    taken += 1
                    tiles, per = -(-rows // (16 * rb)), -(-units // s)
                    assert rb in (1, 2) and (s - 1) * per < units <= s * per
                    assert s == 1 or pairs * s * tiles * 16 * rb <= part_rows
                    assert -(-pairs * s // 8) * tiles <= 32
    assert taken > 10000
    assert rules.heads256(1, 400, 15, 2560, 0) == 104 and rules.heads256(8, 400, 15, 10240, 0) == 101 and rules.heads256(16, 400, 15, 32768, 0) == 201
    assert rules.heads256(20, 400, 15, 100000, 0) < 100


# M, N, K -> measured us of what wide_tile takes and on the plain tiles 96 x 96, 128 x 96, 96 x 64
PLAIN_US = [
    ((1323, 1536, 6144), 55.2, (46.1, 42.6, 51.1)),
    ((1323, 1536, 1536), 15.1, (12.9, 15.5, 14.6)),
    ((1600, 720, 960), 9.2, (9.6, 11.5, 8.0)),
    ((1600, 720, 2048), 13.8, (14.3, 16.7, 12.0)),
    ((2000, 1536, 6144), 59.6, (60.3, 48.4, 73.2)),
    ((408, 1536, 6144), 24.4, (42.5, 39.5, 29.4)),
    ((816, 1024, 4096), 15.6, (23.5, 26.7, 18.5)),
    ((1323, 6144, 1536), 29.7, (42.8, 50.5, 43.8)),
    ((6301, 8, 112), 3.5, (9.9, 9.9, 3.8)),  # (of these three 96 x 64 alone was timed)
    ((7527, 32, 96), 3.6, (9.9, 9.9, 3.9)),
    ((1330, 32, 128), 3.6, (9.9, 9.9, 3.8)),
]


@pytest.mark.parametrize("shape,wide,plain", PLAIN_US)
def test_plain_tiles_are_taken_where_they_are_faster(rules, shape, wide, plain):
    t = rules.plain(*shape)
    took = wide if t < 6 else plain[t - 6]
    assert took <= 1.05 * min(plain + (wide,))


def test_a_plain_tile_is_named_for_every_size(rules):
    for M in (1, 33, 512, 513, 1323, 4000, 18944, 1 << 20):
        for N in (8, 64, 720, 1536, 8192, 151936):
            for K in (16, 960, 6144, 1 << 20):
                t = rules.plain(M, N, K)
                assert -1 <= t < 9
                if t < 6:
                    assert t == rules.wide(M, N, K, 0)


def test_128_wide_heads_leave_the_staged_tiles_beyond_one_workgroup_a_cu(rules):
    """... unless the caches are unaligned or the override pins the staged tiles."""
    assert [rules.ring128(w, 1, -1) for w in (1, 255, 256, 257, 1020)] == [0, 0, 0, 1, 1]
    assert not rules.ring128(1020, 0, -1) and not rules.ring128(1020, 1, 0) and rules.ring128(1020, 1, 1)


# (observation, kv head) pairs, query rows, keys -> measured us of the tiled kernel with its merge launch and of the 256-wide kernel
HEADS_US = [((1, 400, 955), 16.6, 10.8), ((8, 400, 955), 21.9, 16.2), ((16, 400, 955), 27.8, 21.9),
            ((1, 8, 523), 8.8, 9.8), ((1, 16, 523), 9.6, 10.3), ((2, 8, 700), 10.9, 11.6), ((1, 32, 400), 9.7, 10.1), ((6, 32, 400), 11.8, 12.3), ((16, 8, 955), 14.5, 12.6),
            ((32, 128, 1990), 31.1, 72.7), ((64, 64, 1990), 38.0, 78.4), ((24, 256, 1990), 32.6, 53.2), ((48, 64, 955), 21.1, 25.6), ((24, 128, 1990), 26.5, 36.9),
            ((16, 256, 3000), 32.1, 47.1), ((12, 400, 3000), 53.1, 57.5), ((8, 400, 3000), 27.1, 32.5), ((6, 400, 1990), 22.4, 26.2), ((1, 400, 1990), 50.2, 17.6),
            ((64, 8, 1990), 37.9, 30.6)]


@pytest.mark.parametrize("shape,tiled,wide", HEADS_US)
def test_256_wide_heads_take_the_faster_kernel(rules, shape, tiled, wide):
    """... also where an XCD's L2 does not hold the K and V^T that its row tiles share, and where few rows leave the wavefronts idle."""
    pairs, rows, keys = shape
    took = wide if rules.heads256(pairs, rows, -(-keys // 64), 1 << 20, 0) >= 100 else tiled
    assert took <= 1.04 * min(tiled, wide)
