"""The size of the fix-up list (cupf_amd/csrc/capacity.h): a grid without a
strip gets no more than its interior and the rounding of the 64 shares, a strip
no more than its waves' rows on top, and segment offsets stay whole where the
list passes 32 bits.  (That every point finds room is
tests/test_fix_segments_cpu.py.)  Compiled with g++ on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "capacity.h"
using namespace cupf;
int main() {
    int bad = 0;
    const int grids[][3] = {{18, 40, 40}, {35, 35, 35}, {99, 99, 131}, {66, 66, 66}, {130, 50, 300}, {82, 4, 4000},
                            {20, 1000, 90}};  // no strip
    for (auto& g : grids) {
        const long long rows = (long long)(g[1] - 2) * (g[2] - 2), cap = 64 * fix_segment_cap(g[0], g[1], g[2], 16, 64);
        const bool ok = cap >= worst_fix_entries(g[0], g[1], g[2]) && cap <= (rows + 63) * (g[0] - 2);
        if (!ok) std::printf("%d x %d x %d: %lld\n", g[0], g[1], g[2], cap);
        bad += !ok;
    }
    // strips: (67^3: 1 column, 64 rows to a wave) the tiles' points and a wave's rows for one y row of each share
    const long long c67 = 64 * fix_segment_cap(67, 67, 67, 16, 64);
    bad += c67 > 64LL * (67 * 64 + 65 * 64);
    bad += 64 * fix_segment_cap(12, 4, 30, 16, 64) > 64 * 10 * 2;  // two rows, not the six that a wave could hold
    // a list past 32 bits: the last segment's offset
    const long long cap = fix_segment_cap(4, 66, 1600000, 16, 64);
    bad += 64 * cap <= 1LL << 32 || cap >= 1LL << 32;
    for (int shift = 0; shift <= 6; ++shift) {
        const int last = (64 >> shift) - 1;
        bad += (long long)fix_segment_base(last, shift, (unsigned)cap) != 64 * cap - (cap << shift);
        bad += fix_segment_cap(4, 66, 1600000, 16, 64 >> shift) != cap << shift;
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
"""


def test_fix_list_is_no_larger_than_its_points(tmp_path):
    src = tmp_path / "size.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "size"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "cupf_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
