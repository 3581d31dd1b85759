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
