"""The device bytes that a served request is admitted with
(cupf_amd/ensemble.py) against the sizes that pf_create allocates
(cupf_amd/csrc/capacity.h, compiled with g++ on the CPU): a context's large
arrays element for element, over grids with and without a strip, and never less
in all than those arrays hold."""
import os
import subprocess

from cupf_amd import ensemble

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GRIDS = ensemble.GRIDS + [(16, 16, 16), (14, 90, 20), (2, 61, 300), (64, 64, 70), (128, 128, 128), (63, 40, 24),
                          (70, 9, 16), (256, 256, 512), (16, 40, 12)]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "capacity.h"
int main(int argc, char** argv) {
    for (int q = 1; q + 4 < argc; q += 5) {
        const cupf::ContextSizes s = cupf::context_sizes(std::atoi(argv[q]) + 3, std::atoi(argv[q + 1]) + 3,
            std::atoi(argv[q + 2]) + 3, std::atoi(argv[q + 3]), std::atoi(argv[q + 4]), 16);
        std::printf("%lld %lld %lld %lld %lld %lld\n", s.slots, s.field, s.fix, s.act, s.row, s.items);
    }
}
"""


def test_footprint_counts_what_a_context_allocates(tmp_path):
    src = tmp_path / "sizes.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "sizes"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "cupf_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    for K, depth in ((5, 1), (8, 1), (8, 2)):
        args = [str(v) for n in GRIDS for v in (*n, K, depth)]
        r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=60, check=True)
        assert len(r.stdout.splitlines()) == len(GRIDS)
        for n, line in zip(GRIDS, r.stdout.splitlines()):
            slots, field, fix, act, row, items = (int(v) for v in line.split())
            want = dict(slots=slots, field=field, fix=fix, act=act, row=row, items=items)
            assert ensemble._context_sizes(n, K, depth) == want, n
            spec = ensemble.SimSpec(n=n, seed=1, G=1.0, R=0.1, nsteps=10, grains=6)
            if depth == 1:
                held = 16 * slots + 12 * field + 4 * fix + 8 * act + 8 * row + 12 * items
                assert spec.footprint(K) >= held, n
