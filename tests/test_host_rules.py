"""CPU checks of csrc/host_rules.h, built here with the host compiler."""

from __future__ import annotations

import ctypes
import math
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "skmetal_amd" / "csrc"

SOURCE = r"""
#include "host_rules.h"
#include <set>
using namespace skm;

// A workspace of five buffers whose allocation number `fails` fails: once, then
// again without a failure.  0, or the number of the check that does not hold.
extern "C" int workspace(int fails)
{
    std::set<void*> held;
    int at = 0;
    static char mem[16];
    auto grab = [&](void** p, size_t bytes) {
        if (at++ == fails) return 5;
        *p = mem + bytes;
        held.insert(*p);
        return 0;
    };
    auto drop = [&](void* p) { held.erase(p); };
    void* p[5] = {};
    auto all = [&] { return grab_all({{&p[0], 1}, {&p[1], 2}, {&p[2], 3}, {&p[3], 4}, {&p[4], 5}}, grab, drop); };
    if (fails < 5) {
        if (all() != 5) return 1;
        if (!held.empty()) return 2;
        for (void* q : p)
            if (q != nullptr) return 3;
    }
    fails = -1;
    if (all() != 0) return 4;
    if (held.size() != 5) return 5;
    for (int i = 0; i < 5; ++i)
        if (p[i] != mem + i + 1) return 6;
    return 0;
}
extern "C" bool lost(long n, int ld, int k, long left, long passes) { return screen_lost(n, ld, k, left, passes); }
extern "C" long rows(long n, int k) { return wide_rows(n, k); }
extern "C" long blocks(long rows, int k) { return wide_blocks(rows, k); }
extern "C" long part_bytes(long rows, int k) { return (long)wide_part_floats(rows, k) * 4; }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(d / "rules.cpp"),
                    "-o", str(d / "rules.so")], check=True)
    lib = ctypes.CDLL(str(d / "rules.so"))
    lib.lost.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_long]
    lib.lost.restype = ctypes.c_bool
    for f in (lib.rows, lib.blocks, lib.part_bytes):
        f.argtypes, f.restype = [ctypes.c_long, ctypes.c_int], ctypes.c_long
    return lib


@pytest.mark.parametrize("fails", range(6))
def test_a_workspace_is_whole_or_absent(rules, fails):
    assert rules.workspace(fails) == 0


# all rows in one launch: 4.8 and 5.1 G threads, where HIP takes less than 2^32,
# and 38 and 41 GB of workspace
@pytest.mark.parametrize("n,k", [(100_000_000, 6_000), (10_000_000, 65_536), (2**31 - 1, 2**20), (2**31 - 1, 129),
                                 (300, 2**20), (2048, 257), (1, 1), (212_000, 20_000)])
def test_the_wide_screen_in_launches_that_hip_takes(rules, n, k):
    rows = rules.rows(n, k)
    assert 0 < rows <= n and (rows == n or rows % 2048 == 0)
    assert rules.blocks(rows, k) * 512 < 2**32 and (rows + 255) // 256 * 256 < 2**32
    assert rules.part_bytes(rows, k) == rows * ((k + 255) // 256) * 16 <= 2**28
    # (the rows of a launch: their blocks cover them, 256 a block and 256 centres)
    assert rules.blocks(rows, k) * 256 >= rows * ((k + 255) // 256)


# what steps took without and with the screen (us), the rows left evenly over X,
# where the two differ by about a tenth or more
@pytest.mark.parametrize("n,ld,k,share,plain,screened", [
    (1_000_000, 128, 256, 0.4, 340, 260), (1_000_000, 128, 256, 0.9, 339, 416), (250_000, 128, 256, 0.2, 95, 70),
    (250_000, 128, 256, 0.6, 95, 106), (1_000_000, 64, 1024, 0.6, 650, 543), (1_000_000, 64, 1024, 0.9, 640, 716),
    (120_000, 64, 1024, 0.2, 98, 86), (120_000, 64, 1024, 0.5, 98, 116), (300_000, 32, 1024, 0.3, 136, 100),
    (200_000, 128, 2048, 0.6, 562, 489), (200_000, 128, 2048, 0.9, 563, 628), (400_000, 300, 200, 0.2, 329, 290),
    (400_000, 300, 200, 0.5, 330, 399), (64_000, 768, 400, 0.3, 215, 194), (64_000, 768, 400, 0.6, 216, 302),
    (130_000, 512, 512, 0.4, 297, 273), (130_000, 512, 512, 0.6, 301, 351), (100_000, 768, 2048, 0.6, 1511, 1270),
    (8_000, 768, 1500, 0.9, 541, 176), (20_000, 400, 600, 0.9, 156, 112), (390_000, 768, 200, 0.2, 643, 510),
    (390_000, 768, 200, 0.6, 647, 750), (50_000, 200, 1000, 0.2, 136, 118), (50_000, 200, 1000, 0.6, 137, 159),
    (30_000, 1000, 200, 0.5, 134, 109), (30_000, 1000, 200, 0.9, 135, 155), (500_000, 768, 4096, 0.6, 13760, 12227),
    (500_000, 768, 4096, 0.8, 13773, 15280), (300_000, 768, 2048, 0.6, 4336, 3706), (1_000_000, 300, 2000, 0.5, 5743, 4901),
    (1_000_000, 300, 2000, 0.8, 5762, 6727), (200_000, 1000, 1000, 0.7, 2214, 1947), (1_000_000, 200, 600, 0.3, 1470, 1196),
    (1_000_000, 200, 600, 0.6, 1455, 1681), (300_000, 512, 1024, 0.5, 1430, 1260), (300_000, 512, 1024, 0.8, 1392, 1606),
    (4_000_000, 64, 1024, 0.6, 2641, 2101), (4_000_000, 64, 1024, 0.9, 2594, 2837), (2_000_000, 128, 1000, 0.6, 2429, 2003),
    (2_000_000, 128, 1000, 0.9, 2362, 2682),
])
def test_the_screen_is_kept_where_it_was_faster(rules, n, ld, k, share, plain, screened):
    block = ((n + 255) // 256 + 63) // 64 * 64  # rows of a block's share
    busiest = share * block + 2.8 * math.sqrt(share * (1 - share) * block)  # of 256 blocks
    assert rules.lost(n, ld, k, int(share * n), math.ceil(busiest / 256)) == (screened > plain)


def test_rows_left_in_one_stretch(rules):
    # a tenth of 1M x 128: 338 without the screen, 404 with it
    assert rules.lost(1_000_000, 128, 256, 100_000, 16)
    assert not rules.lost(1_000_000, 128, 256, 100_000, 2)
