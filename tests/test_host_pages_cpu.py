"""Pages of result buffers (cupf_amd/csrc/host_pages.h): made present where they
are absent, contents kept, and no thread taken for buffers that are small or
whose pages are there.  Compiled with g++ on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include "host_pages.h"
using namespace cupf;
static char* fresh(size_t n) {
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    return p == MAP_FAILED ? nullptr : (char*)p;
}
static size_t absent(char* p, size_t n) {  // p page-aligned
    std::vector<unsigned char> v((n + kHostPage - 1) / kHostPage);
    if (mincore(p, n, v.data()) != 0) return 1u << 30;
    size_t c = 0;
    for (unsigned char b : v) c += !(b & 1);
    return c;
}
int main() {
    int bad = 0;
    auto want = [&](bool ok, const char* what) { if (!ok) { ++bad; std::printf("%s\n", what); } };
    for (size_t n : {size_t(8) << 20, (size_t(9) << 20) + 12345, (size_t(33) << 20) + 4}) {
        char* p = fresh(n);
        char* q = fresh(n);
        if (!p || !q) return 2;
        p[n / 2] = 7;
        const bool advised = madvise(q, kHostPage, 23) == 0;  // the kernel knows the advice
        want(make_present({{p + 4, n - 4}, {nullptr, n}}) > 0 || n - 4 < (size_t(8) << 20), "a fresh buffer was left");
        if (n - 4 >= (size_t(8) << 20) && advised) want(absent(p + kHostPage, n - 2 * kHostPage) == 0, "pages left absent");
        want(p[n / 2] == 7 && p[n / 2 + 1] == 0, "contents changed");
        std::memset(p, 1, n);
        std::memset(q, 2, n);
        want(make_present({{p, n}, {q, n}}) == 0, "threads for pages that are there");
        madvise(q + (n - (size_t(1) << 20)) / kHostPage * kHostPage, size_t(1) << 20, MADV_DONTNEED);
        want(make_present({{p, n}, {q, n}}) > 0, "an absent end was left");
        want(p[0] == 1 && p[n - 1] == 1 && q[0] == 2, "contents changed");
        munmap(p, n);
        munmap(q, n);
    }
    char* s = fresh(4 << 20);
    want(make_present({{s, size_t(4) << 20}}) == 0, "threads for a small buffer");
    return bad;
}
"""


def test_only_absent_pages_of_large_buffers_take_threads(tmp_path):
    src = tmp_path / "pages.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "pages"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "cupf_amd", "csrc"), str(src), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
