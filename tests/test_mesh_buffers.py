"""The triangle-mesh passes' buffers when an allocation fails while they grow: they must not go
on claiming the size they had, since what failed was freed. The host side of the header is
compiled with an allocator of the test's own that refuses from a given call on; no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "pgx_internal.h"
#include <cstdio>
#include <cstdlib>
static int left = 1 << 30;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    if (left-- <= 0) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::malloc(n);
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
int main() {
    for (int hulls = 0; hulls < 2; ++hulls)
        for (int ok = 0; ok < 8; ++ok) {
            pgx::MeshBuffers b;
            left = 1 << 30;
            b.reserve(4, 16, hulls != 0);
            left = ok;
            bool failed = false;
            try { b.reserve(8, 32, hulls != 0); } catch (...) { failed = true; }
            left = 1 << 30;
            b.reserve(8, 16, hulls != 0);   // as the next call asks again
            const bool whole = b.cand.p && b.pairOf.p && b.recs.p && b.candOff.p && b.candCount.p &&
                               (!hulls || (b.hitList.p && b.simplex.p));
            const size_t cap = (size_t)b.candCap;
            const bool sizes = cap >= 16 && b.cand.n >= cap && b.pairOf.n >= cap && b.recs.n >= 15 * cap &&
                               (!hulls || (b.hitList.n >= cap && b.simplex.n >= 36 * cap));
            std::printf("%d %d %d %d\n", hulls, ok, failed ? 1 : 0, whole && sizes ? 1 : 0);
        }
}
"""


def test_a_failed_growth_leaves_no_stale_size(tmp_path):
    from physecs_amd import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "buffers.hip", tmp_path / "buffers"
    src.write_text(PROGRAM)
    subprocess.run([build.HIPCC, "--offload-host-only", "-O0", "-std=c++17", "-w", "-I",
                    os.path.join(ROOT, "physecs_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src), "-o",
                    str(exe)], check=True, capture_output=True, timeout=300)
    rows = [tuple(map(int, x.split())) for x in
            subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()]
    assert len(rows) == 16
    for hulls, ok, failed, whole in rows:
        assert failed == (ok < (7 if hulls else 5)) and whole, (hulls, ok)
