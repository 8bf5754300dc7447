"""Host-side check of the rule that sends a plain step to 16 lanes per agent
(csrc/row_rule.h, compiled with g++; nothing runs on a GPU): the grid's size
covers every count, follows a crowd that grows or shrinks by much and stays
where it is while the count moves around any value; no crowd takes the form
past the limit of its k, whatever it was before."""
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
        r.update(true, 10, at + 60);
        r.update(true, 10, at - 60);
        const int settled = r.agents;
        for (int i = 0; i < 40; ++i) {
            const int n = at - 60 + rnd(121);
            r.update(true, 10, n);
            moves += r.agents != settled;
            short_of += r.agents < n;
        }
    }
    ecm::RowRule r;
    for (int i = 0; i < 20000; ++i) {
        const int n = rnd(i % 7 == 0 ? 90000 : 9000);
        r.update(true, 10, n);
        short_of += r.agents < n;
        const int spare = r.agents - n;
        too_large += spare > 8192 && spare > r.agents / 4;
    }
    r.update(false, 10, 100);
    printf("%ld %ld %ld %d\n", short_of, too_large, moves, r.agents);
    return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="g++ not found")
def test_grid_size_covers_the_crowd_and_keeps_still():
    assert run("#include <cstdint>\n" + GRID) == [0, 0, 0, 0]


LIMITS = r"""
#include "row_rule.h"
#include <cstdio>
#include <cstdlib>
int main(int, char** v) {
    const int k = atoi(v[1]), limit = atoi(v[2]);
    auto form = [&](int first, int then) {
        ecm::RowRule r;
        if (first) r.update(true, k, first);
        r.update(true, k, then);
        return (int)r.step;
    };
    const int back = limit - limit / 8;
    printf("%d %d %d %d %d %d ", form(0, limit), form(0, limit + 1), form(limit - 1, limit + 1), form(1, 2 * limit),
           form(limit + 1, back + 1), form(limit + 1, back));
    // a step in another shape, or a learned one, does not count as a crowd past the limit
    ecm::RowRule r;
    r.update(false, k, limit);
    printf("%d ", (int)r.step);
    r.update(true, k, limit);
    printf("%d ", (int)r.step);
    // the attraction pass: its own limit
    ecm::RowRule a;
    for (int n : {16000, 16001, 14001, 14000}) {
        a.update(true, k, n);
        printf("%d ", (int)a.attr);
    }
    return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="g++ not found")
@pytest.mark.parametrize("k,limit", [(1, 112000), (5, 112000), (6, 160000), (10, 160000), (11, 200000), (16, 200000)])
def test_no_crowd_past_its_limit_takes_the_form(k, limit):
    assert run(LIMITS, k, limit) == [1, 0, 0, 0, 0, 1, 0, 1, 1, 0, 0, 1]
