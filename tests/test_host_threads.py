"""Host work on threads when memory runs out: a thread that cannot be started
leaves its share to the others, whichever allocation fails."""
import os
import subprocess

import chysx

HOST = os.path.join(os.path.dirname(os.path.dirname(chysx.__file__)), "csrc", "host")

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "threads.h"

static std::atomic<long> countdown{-1};
void* operator new(std::size_t n) {
    if (countdown.load() >= 0 && countdown.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
    for (long fail = 0; fail < 32; ++fail) {
        std::atomic<int> sum{0};
        countdown = fail;
        chysx::for_each_on_threads(100, 8, [&](std::size_t i) { sum += int(i); });
        countdown = -1;
        if (sum != 4950) return 1;
    }
    int caught = 0;
    try {
        chysx::for_each_on_threads(100, 8, [&](std::size_t i) { if (i == 50) throw 7; });
    } catch (int e) {
        caught = e;
    }
    return caught == 7 ? 0 : 2;
}
"""


def test_threads_that_cannot_start_leave_their_work_to_the_others(tmp_path):
    src, exe = tmp_path / "threads.cpp", tmp_path / "threads"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", HOST, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
