"""CPU checks of csrc/host_rules.h, built here with the host compiler."""

from __future__ import annotations

import ctypes
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
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(d / "rules.cpp"),
                    "-o", str(d / "rules.so")], check=True)
    return ctypes.CDLL(str(d / "rules.so"))


@pytest.mark.parametrize("fails", range(6))
def test_a_workspace_is_whole_or_absent(rules, fails):
    assert rules.workspace(fails) == 0
