"""The pool of freed device blocks on the host, with the HIP calls it makes replaced by ones that keep count.

What it holds and what it frees when host memory runs out at any point of taking a block in, and when a block is
larger than all it may hold."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omm-bundle_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include <set>

#include "omx_pool.h"

static std::set<void *> freed;
static long allocations_left = -1;  // of host memory until one fails; -1: none does
static size_t device_bytes = (size_t)1 << 40;

void *operator new(size_t n) {
    if (allocations_left == 0) throw std::bad_alloc();
    if (allocations_left > 0) --allocations_left;
    if (void *p = malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" hipError_t hipFree(void *p) {
    const long left = allocations_left;
    allocations_left = -1;
    if (!freed.insert(p).second) printf("freed twice\n");
    allocations_left = left;
    return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
extern "C" hipError_t hipMemGetInfo(size_t *avail, size_t *total) { return *avail = *total = device_bytes, hipSuccess; }

using omx::DevPool;
static void *at(int q) { return (void *)(size_t)(4096 * (q + 1)); }
static bool idle(DevPool &pool, int q) {
    size_t b;
    int d;
    return pool.claim(at(q), b, d) == DevPool::IDLE;
}
static void put(DevPool &pool, int q, size_t bytes) {
    size_t b;
    int d;
    pool.note(at(q), bytes);
    if (pool.claim(at(q), b, d) != DevPool::LIVE || b != bytes) printf("block %d not live\n", q);
    pool.put(at(q), b, d);
}

static void out_of_host_memory() {
    int whole = 0;
    for (int n = 0; n < 12; ++n) {
        DevPool pool;
        freed.clear();
        for (int q = 0; q < 64; ++q) put(pool, q, 1000 + q);
        size_t b;
        int d;
        pool.note(at(64), 2000);
        pool.claim(at(64), b, d);
        bool threw = false;
        allocations_left = n;
        try {
            pool.put(at(64), b, d);
        } catch (const std::bad_alloc &) {
            threw = true;
        }
        allocations_left = -1;
        whole += !threw;
        // thrown: nothing has changed, the caller frees the block; else the oldest made room for it
        for (int q = 0; q < 64; ++q)
            if (idle(pool, q) == (!threw && q == 0) || freed.count(at(q)) != (!threw && q == 0)) printf("after %d: block %d\n", n, q);
        if (idle(pool, 64) == threw || freed.count(at(64))) printf("after %d: the new block\n", n);
    }
    if (whole < 6) printf("put needs too many allocations\n");
}

static void large_blocks() {
    device_bytes = 64 * 1000;  // 1001 bytes are kept
    DevPool pool;
    for (int q = 0; q < 3; ++q) put(pool, q, 300);
    put(pool, 3, 5000);
    for (int q = 0; q < 3; ++q)
        if (!idle(pool, q)) printf("block %d gone\n", q);
    if (idle(pool, 3) || freed != std::set<void *>{at(3)}) printf("the large block stays\n");
    put(pool, 4, 300);
    if (idle(pool, 0) || !idle(pool, 1) || !idle(pool, 2) || !idle(pool, 4)) printf("the oldest did not go\n");
    put(pool, 5, 1001);
    if (!idle(pool, 5) || idle(pool, 1) || idle(pool, 2) || idle(pool, 4)) printf("a block of the whole room\n");
}

int main(int, char **argv) {
    if (argv[1][0] == 'm') out_of_host_memory();
    if (argv[1][0] == 'l') large_blocks();
    printf("done\n");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "pool.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-o",
                    str(d / "pool"), str(d / "pool.cpp")], check=True)
    return str(d / "pool")


def _run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "done\n"), r.stdout


def test_host_memory_runs_out(program):
    _run(program, "memory")


def test_large_block_leaves_the_others(program):
    _run(program, "large")
