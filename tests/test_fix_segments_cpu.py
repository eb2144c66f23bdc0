"""The fix-up list's segments (cupf_amd/csrc/capacity.h) against a brute-force
placement of every interior point of small grids: no segment can receive more
points than it holds, whatever the split, and every split uses the full
list.  Compiled with g++ on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <map>
#include <vector>
#include "capacity.h"
using namespace cupf;
int main() {
    const std::vector<std::vector<int>> grids = {{5, 5, 5}, {19, 12, 30}, {67, 67, 20}, {66, 9, 40}, {82, 81, 20},
        {130, 11, 17}, {259, 13, 70}, {34, 34, 34}, {98, 98, 30}, {4, 200, 50}, {17, 90, 33}, {81, 70, 9},
        {70, 3, 90}, {131, 4, 3}, {66, 300, 5}, {75, 64, 64}};
    int bad = 0;
    for (auto& g : grids)
        for (int S = 1; S <= 64; S *= 2) {
            const int fnx = g[0], fny = g[1], fnz = g[2];
            const int tiles = cap_tiles_x(fnx, 16), ex = (fnx - 2) - 64 * tiles;
            std::map<long long, long long> points;
            for (int k = 1; k <= fnz - 2; ++k)
                for (int j = 1; j <= fny - 2; ++j)
                    for (int i = 1; i <= fnx - 2; ++i) {
                        // the first y row of the wave that holds the point
                        const int per = 64 / std::max(ex, 1);
                        const int first = (i - 1) / 64 < tiles ? j : 1 + (j - 1) / per * per;
                        ++points[((first - 1) * (fnz - 2) + k - 1) / (((fny - 2) * (fnz - 2) + 63) / 64) * S / 64];
                    }
            const long long cap = fix_segment_cap(fnx, fny, fnz, 16, S);
            const long long all = 64 * fix_segment_cap(fnx, fny, fnz, 16, 64);
            for (auto& p : points) bad += p.second > cap || p.first < 0 || p.first >= S;
            bad += S * cap != all || all < worst_fix_entries(fnx, fny, fnz);
        }
    std::printf("%d mismatches\n", bad);
    return bad != 0;
}
"""


def test_segments_hold_their_rows(tmp_path):
    src = tmp_path / "seg.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "seg"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "cupf_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
