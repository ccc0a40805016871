"""The device-memory arena (sw_memory.hpp) on a stub device of a few megabytes,
and the blocks that one gradient keeps for the next on the device itself."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import cases
import harness
from simwave_amd import adjoint
from simwave_amd import build as hipbuild
from simwave_amd.device import DeviceForward

CSRC = os.path.join(harness.REPO, "simwave_amd", "csrc")

# A device of CAP bytes: freed memory goes to a pool (reusable by a request of
# at most its size, smallest first) and only a trim after a synchronisation
# makes it free memory again.
STUB = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>
#include "sw_memory.hpp"
static const size_t MB = 1u << 20, CAP = 64 * MB;
static std::map<void *, size_t> live, pool, done, kept;
static std::vector<void *> order;          // kept blocks, oldest first
static size_t total(const std::map<void *, size_t> &m)
{
    size_t s = 0;
    for (auto &x : m) s += x.second;
    return s;
}
struct Full {};
static size_t bound = 0;
struct Stub {
    typedef int stream;
    static int device() { return 0; }
    static bool alloc(void **p, size_t bytes, int)
    {
        static size_t next = 4096;
        for (auto *m : {&pool, &done})
            for (auto &x : *m)
                if (x.second == bytes) {
                    *p = x.first;
                    live[*p] = bytes;
                    m->erase(*p);
                    return true;
                }
        if (total(live) + total(pool) + total(done) + total(kept) + bytes > CAP) return false;
        *p = (void *)(next += 4096);
        live[*p] = bytes;
        return true;
    }
    static void free(void *p, int)
    {
        if (!live.count(p)) abort();
        pool[p] = live[p];
        live.erase(p);
    }
    static bool synchronize(int) { done.insert(pool.begin(), pool.end()); pool.clear(); return true; }
    static void trim() { done.clear(); }
    static void *take(int, size_t bytes, size_t *got)
    {
        for (size_t i = 0; i < order.size(); i++) {
            void *p = order[i];
            if (kept[p] >= bytes && kept[p] - bytes <= bytes / 4) {
                *got = live[p] = kept[p];
                kept.erase(p);
                order.erase(order.begin() + i);
                return p;
            }
        }
        return nullptr;
    }
    static bool put(int, void *p, size_t bytes, size_t)
    {
        if (live[p] != bytes) abort();
        live.erase(p);
        kept[p] = bytes;
        order.push_back(p);
        return true;
    }
    static void *evict(int, size_t limit)
    {
        if (total(kept) <= limit) return nullptr;
        void *p = order.front();
        order.erase(order.begin());
        live[p] = kept[p];
        kept.erase(p);
        return p;
    }
    [[noreturn]] static void out_of_memory(size_t) { throw Full{}; }
    static size_t limit() { return bound; }
    [[noreturn]] static void region_full(size_t, size_t, size_t) { throw Full{}; }
};
typedef sw::Arena<Stub> Arena;
static void gradient(std::vector<size_t> mb)
{
    Arena a(0);
    a.keep_blocks();
    for (size_t m : mb) a.alloc<char>(m * MB);
}
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
int main()
{
    gradient({20, 20});                      // leaves 40 MB in kept blocks
    CHECK(total(kept) == 40 * MB && live.empty());
    gradient({18, 20});                      // served from them
    CHECK(total(kept) == 40 * MB && order.size() == 2);
    {
        Arena a(0);                          // a forward that needs their memory
        a.alloc<char>(50 * MB);
        CHECK(total(kept) == 0);
    }
    CHECK(live.empty());
    Stub::synchronize(0); Stub::trim();
    gradient({20, 20});
    {
        void *p = Arena::fresh(60 * MB, 0);  // the memory entry point
        CHECK(live.size() == 1 && live.count(p) && total(kept) == 0);
        Stub::free(p, 0);
    }
    Stub::synchronize(0);                    // the pool alone holds the memory
    CHECK(total(done) == 60 * MB && total(kept) == 0);
    {
        Arena a(0);
        a.alloc<char>(30 * MB);
        CHECK(total(done) == 0);
    }
    Stub::synchronize(0); Stub::trim();
    {
        Arena a(0);                          // blocks the run itself released
        a.keep_blocks();
        void *p = a.alloc<char>(40 * MB), *q = a.alloc<char>(20 * MB);
        a.release(p);
        CHECK(a.alloc<char>(36 * MB) == p);  // in order on one stream
        a.release(p);
        CHECK(a.alloc<char>(42 * MB) != q && live.size() == 2);
        a.alloc<char>(100);                  // a small request of a keeping arena
    }
    CHECK(live.empty() && total(kept) == 62 * MB);
    {
        Arena a(0);
        a.keep_blocks();
        a.alloc<char>(62 * MB);              // no block fits: all of them go first
    }
    bool full = false;
    try { Arena a(0); a.alloc<char>(10 * MB); a.alloc<char>(60 * MB); } catch (Full) { full = true; }
    CHECK(full && live.empty() && total(kept) == 0);
    bound = 4 * MB;                          // a bound on one run
    full = false;
    try { Arena a(0); a.alloc<char>(3 * MB); a.alloc<char>(2 * MB); } catch (Full) { full = true; }
    CHECK(full && live.empty());
    bound = 0;
    char region[1024];
    Arena r(0, region, sizeof region);       // a caller's region
    CHECK(r.alloc<char>(1) == region && r.alloc<float>(64) == (float *)(region + 256));
    full = false;
    try { r.alloc<char>(513); } catch (Full) { full = true; }
    CHECK(full && r.alloc<char>(512) == region + 512);
    printf("ok\n");
    return 0;
}
"""


def test_memory_held_back_is_given_back_when_the_device_is_full(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    src, exe = tmp_path / "arena.cpp", tmp_path / "arena"
    src.write_text(STUB)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.stdout == "ok\n" and res.returncode == 0, res.stdout


@pytest.mark.gpu
def test_second_gradient_takes_the_blocks_of_the_first():
    import torch
    print("kept blocks taken", flush=True)
    held = ctypes.CDLL(hipbuild.common_library_path())["simwave_hip_block_held"]
    held.restype, held.argtypes = ctypes.c_ulonglong, [ctypes.c_int]
    _, solver, kw = cases.adjoint_shot("3d_so8", dtype=np.float32, shape=(60, 64, 70))
    rr = np.ones((kw["end_timestep"], kw["num_receivers"]), np.float32)
    lib = DeviceForward(solver, buffers="torch")._lib
    assert lib.simwave_hip_trim_pool() == 0 and held(torch.cuda.current_device()) == 0
    first = adjoint.gradient(solver, rr, checkpoint_every=4)["grad_velocity"]
    kept = held(torch.cuda.current_device())
    assert kept >= 10 * 4 * 60 * 64 * 70
    second = adjoint.gradient(solver, rr, checkpoint_every=4)["grad_velocity"]
    assert held(torch.cuda.current_device()) == kept      # fresh ones would double it
    np.testing.assert_array_equal(second, first)
    assert lib.simwave_hip_trim_pool() == 0 and held(torch.cuda.current_device()) == 0
