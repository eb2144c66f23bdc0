"""The range of the epoch counter (cupf_amd/csrc/capacity.h): whatever the
length of a batched call and wherever the counter stands, an epoch shifted by
the 4 bits of a row word's bound stays within 32 bits, and no step is lost.
Compiled with g++ on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "capacity.h"
using namespace cupf;
// one batched call, as pf_batch_step makes it: runs, a renewal ahead of a run
// whose epochs do not fit (both buffers' maps take one each), an epoch per step
// and the next step's that the last one leaves
static bool call(unsigned ctr, int nsteps) {
    long long done = 0;
    for (int left = nsteps; left > 0;) {
        const int seg = epoch_run(left);
        if (seg < 1 || seg > left) return false;
        if (!epochs_left(ctr, (unsigned)seg + 2u)) ctr = 3u;
        if ((unsigned long long)ctr + seg + 1u > kEpochMax) return false;
        ctr += (unsigned)seg;
        done += seg;
        left -= seg;
    }
    return done == nsteps && (ctr << 4 >> 4) == ctr;
}
int main() {
    const unsigned at[] = {1u, 3u, 1000u, 1u << 26, kEpochMax / 2, kEpochMax - 402u, kEpochMax - 3u, kEpochMax - 1u,
                           kEpochMax, kEpochMax + 1000u};
    const int steps[] = {1, 2, 8, 400, 1 << 20, (1 << 26) - 1, 1 << 26, (1 << 26) + 1, 134217724, 134217725, 134217726,
                         134217727, 134217728, 200000000, 268435456, 300000000, 1 << 30, 0x7ffffffd, 0x7ffffffe,
                         0x7fffffff};
    int bad = 0, n = 0;
    for (unsigned c : at)
        for (int s : steps) {
            ++n;
            if (!call(c, s)) {
                ++bad;
                std::printf("counter %u, %d steps\n", c, s);
            }
        }
    std::printf("%d calls, %d bad\n", n, bad);
    return bad != 0 || (kEpochMax << 4 >> 4) != kEpochMax;
}
"""


def test_epochs_of_a_long_batched_call_fit_the_row_words(tmp_path):
    src = tmp_path / "epochs.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "epochs"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "cupf_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
