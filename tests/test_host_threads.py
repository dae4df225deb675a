"""csrc/host_threads.hpp on the CPU: work shared among threads is done once each
and ends before the call returns, also where a thread cannot be started (no
threads left, no memory for one) and where some of it throws."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <stdexcept>
#include <pthread.h>

#include "host_threads.hpp"

static std::atomic<int> limit{-1};   // calls on the main thread that still succeed; -1: all
static bool no_memory, no_threads;
static pthread_t main_thread;
static bool fails() { return pthread_equal(pthread_self(), main_thread) && limit >= 0 && limit-- <= 0; }

void* operator new(std::size_t n) {
    if (no_memory && fails()) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" int __real_pthread_create(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
extern "C" int __wrap_pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
    if (no_threads && fails()) return EAGAIN;
    return __real_pthread_create(t, a, f, x);
}

int main(int argc, char** argv) {
    main_thread = pthread_self();
    const char* what = argv[1];
    const int n = std::atoi(argv[2]), good = std::atoi(argv[3]);
    std::atomic<int> done[16] = {};
    no_memory = !std::strcmp(what, "memory");
    no_threads = !std::strcmp(what, "threads");
    bool thrown = false;
    if (no_memory) limit = 2 + good;  // the two vectors of the call itself, then a state per thread
    if (no_threads) limit = good;
    try {
        hgdg::on_threads(n, [&](int w) {
            ++done[w];
            if (!std::strcmp(what, "throws") && w == good) throw std::runtime_error("work");
        });
    } catch (const std::runtime_error&) {
        thrown = true;
    }
    limit = -1;
    for (int w = 0; w < 16; ++w)
        if (done[w] != (w < n ? 1 : 0)) return 1;
    return thrown == !std::strcmp(what, "throws") ? 0 : 2;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    folder = tmp_path_factory.mktemp("threads")
    source = folder / "t.cpp"
    source.write_text(SOURCE)
    exe = folder / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "hpgem_amd", "csrc"), str(source),
                    "-pthread", "-o", str(exe), "-static-libstdc++", "-Wl,--wrap=pthread_create"], check=True)
    return str(exe)


@pytest.mark.parametrize("what,n,good", [("none", 1, 0), ("none", 4, 0), ("throws", 4, 0), ("throws", 4, 2),
                                         ("memory", 4, 0), ("memory", 4, 1), ("memory", 4, 2),
                                         ("threads", 4, 0), ("threads", 4, 2)])
def test_on_threads(program, what, n, good):
    assert subprocess.run([program, what, str(n), str(good)], timeout=60).returncode == 0
