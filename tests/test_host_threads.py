"""Host threads of a read-back: where a thread cannot be started, for want of threads
or of memory, the calling thread does its share, and nothing is thrown past the
library's C entry points.  A small host program with an allocator that fails stands
in for the shortage."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mittet_main_amd", "csrc")
PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "host_threads.h"

static std::atomic<int> left{1 << 30};
void *operator new(std::size_t n)
{
    if (left-- <= 0)
        throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main(int, char **argv)
{
    std::atomic<int> ran[8];
    for (auto &r : ran)
        r = 0;
    auto work = [&](int t) { ran[t]++; };
    const int n = std::atoi(argv[1]);
    left = std::atoi(argv[2]);   // allocations that succeed, about one for each thread
    mt::on_threads<8>(n, work);
    left = 1 << 30;
    for (int t = 0; t < 8; ++t)
        if (ran[t] != (t < n ? 1 : 0))
            return 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("threads")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, "-o", str(d / "t"), str(d / "t.cpp")],
                   check=True)
    return str(d / "t")


@pytest.mark.parametrize("allocations", [0, 1, 3, 100])
@pytest.mark.parametrize("n", [1, 2, 8])
def test_every_share_runs_once(program, n, allocations):
    assert subprocess.run([program, str(n), str(allocations)], timeout=60).returncode == 0
