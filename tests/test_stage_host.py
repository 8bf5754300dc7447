"""Host-side check of the staging of host batches (csrc/stage.h, compiled with
g++; nothing runs on a GPU).  A queue that keeps every copy pending until it is
waited for stands for the device: the bytes must arrive whole for sizes around
the pieces, no piece may be filled while its copy is pending, and however a
call ends (a copy that fails, an error after the staging, success), nothing may
be pending once it returned."""
import os
import shutil
import subprocess
import tempfile

import pytest

from conftest import ROOT

GXX = shutil.which("g++")
CSRC = os.path.join(ROOT, "ecmgenerator_amd", "csrc")

SRC = r"""
#include "stage.h"
#include <cstdio>
#include <vector>
struct Queue {
    struct Copy { unsigned char* dst; const unsigned char* src; size_t n; };
    std::vector<Copy> pending;
    long copies = 0, waits = 0, fail_at = -1;
    int copy(void* d, const void* s, size_t n) {
        if (copies++ == fail_at) return -3;
        pending.push_back({(unsigned char*)d, (const unsigned char*)s, n});
        return 0;
    }
    int wait() {
        ++waits;
        for (auto& c : pending) memcpy(c.dst, c.src, c.n);
        pending.clear();
        return 0;
    }
};
constexpr size_t kPiece = 64, kPieces = 4;
// one call: two arrays staged, then an error or the call's own wait
static int call(Queue& q, unsigned char* mem, std::vector<unsigned char>& dst, const std::vector<unsigned char>& src,
                size_t second, bool launch_fails, long* busy) {
    ecm::Stager<Queue> st(q, mem, kPiece, kPieces);
    const size_t first = src.size() - second;
    auto fill = [&](void* to, size_t at, size_t len) {
        for (auto& c : q.pending) *busy += c.src < (unsigned char*)to + len && (unsigned char*)to < c.src + c.n;
        memcpy(to, src.data() + at, len);
    };
    if (int rc = st.put(dst.data(), first, fill)) return rc;
    if (int rc = st.put(dst.data() + first, src.data() + first, second)) return rc;
    if (launch_fails) return -5;
    if (int rc = q.wait()) return rc;
    st.waited();
    return 0;
}
int main() {
    std::vector<unsigned char> mem(kPiece * kPieces);
    long bad = 0, busy = 0, left = 0, extra = 0;
    for (size_t n : {1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 5000})
        for (size_t second : {(size_t)0, (size_t)1, n / 2})
            for (int how = 0; how < 6; ++how) {
                std::vector<unsigned char> src(n), dst(n, 0);
                for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(1 + (i * 7 + how) % 251);
                Queue q;
                if (how >= 2) q.fail_at = how - 2;           // a copy fails
                const int rc = call(q, mem.data(), dst, src, second, how == 1, &busy);
                left += (long)q.pending.size();
                if (how == 0) {
                    bad += rc != 0 || dst != src;
                    extra += q.waits > 1 + q.copies / (long)kPieces;
                } else {
                    bad += rc == 0 && q.copies > q.fail_at && q.fail_at >= 0;
                    bad += how == 1 && rc != -5;
                }
            }
    printf("bad %ld busy %ld left %ld extra %ld\n", bad, busy, left, extra);
    return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="g++ not found")
def test_no_call_ends_with_copies_in_flight():
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "stage.cpp")
        exe = os.path.join(d, "stage")
        with open(src, "w") as f:
            f.write(SRC)
        subprocess.run([GXX, "-O2", "-std=c++17", "-I", CSRC, src, "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        assert r.stdout.split() == ["bad", "0", "busy", "0", "left", "0", "extra", "0"]


RULE = r"""
#include "stage.h"
#include <cstdio>
int main() {
    for (bool first : {true, false})
        for (size_t n : {1, 512, 513, 60000}) printf("%d ", (int)ecm::stage_page_locked(first, n));
    return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="g++ not found")
def test_first_call_of_few_rows_allocates_nothing_page_locked():
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "rule.cpp")
        exe = os.path.join(d, "rule")
        with open(src, "w") as f:
            f.write(RULE)
        subprocess.run([GXX, "-O2", "-std=c++17", "-I", CSRC, src, "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        assert r.stdout.split() == ["0", "0", "1", "1"] + ["1"] * 4
