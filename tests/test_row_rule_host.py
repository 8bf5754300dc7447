"""Host-side check of the rule that sends a plain step to 16 lanes per agent
(csrc/row_rule.h, compiled with g++; nothing runs on a GPU): the grid's size
covers every count, follows a crowd that grows or shrinks by much and stays
where it is while the count moves around any value."""
import os
import shutil
import subprocess
import tempfile

import pytest

from conftest import ROOT

GXX = shutil.which("g++")
CSRC = os.path.join(ROOT, "ecmgenerator_amd", "csrc")


def run(src, *args):
    with tempfile.TemporaryDirectory() as d:
        cpp, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        with open(cpp, "w") as f:
            f.write(src)
        subprocess.run([GXX, "-O2", "-std=c++17", "-I", CSRC, cpp, "-o", exe], check=True)
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        return [int(v) for v in r.stdout.split()]


GRID = r"""
#include "row_rule.h"
#include <cstdio>
int main() {
    long short_of = 0, too_large = 0, moves = 0;
    uint32_t seed = 1;
    auto rnd = [&](int m) { seed = seed * 1664525u + 1013904223u; return (int)((seed >> 8) % (uint32_t)m); };
    // around every multiple of 4,096 and elsewhere: settled after the first two counts
    for (int at = 100; at < 100000; at += at < 20000 ? 61 : 1021) {
        ecm::RowRule r;
        r.update(true, at + 60);
        r.update(true, at - 60);
        const int settled = r.agents;
        for (int i = 0; i < 40; ++i) {
            const int n = at - 60 + rnd(121);
            r.update(true, n);
            moves += r.agents != settled;
            short_of += r.agents < n;
        }
    }
    ecm::RowRule r;
    for (int i = 0; i < 20000; ++i) {
        const int n = rnd(i % 7 == 0 ? 90000 : 9000);
        r.update(true, n);
        short_of += r.agents < n;
        const int spare = r.agents - n;
        too_large += spare > 8192 && spare > r.agents / 4;
    }
    r.update(false, 100);
    printf("%ld %ld %ld %d\n", short_of, too_large, moves, r.agents);
    return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="g++ not found")
def test_grid_size_covers_the_crowd_and_keeps_still():
    assert run("#include <cstdint>\n" + GRID) == [0, 0, 0, 0]
