"""The pool of device blocks (device_pool.hpp) against a runtime of two devices that only counts: what it keeps,
when it gives it back, and that it gives all of it back when asked."""
import os
import subprocess

import pytest

from conftest import ROOT

RUNTIME = r'''
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
extern bool no_memory;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipHostMallocPortable = 1 };
struct Runtime {
    int dev = 0;
    std::map<void*, std::pair<int, size_t>> held;
    size_t on(int d) const { size_t s = 0; for (auto& [p, x] : held) if (x.first == d) s += x.second; return s; }
};
inline Runtime& rt() { static Runtime r; return r; }
inline hipError_t hipGetDevice(int* d) { *d = rt().dev; return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) {
    static char* next = reinterpret_cast<char*>(4096);  // addresses only
    const bool m = no_memory; no_memory = false;  // the runtime's own
    *p = next; next += 4096; rt().held[*p] = {rt().dev, n}; no_memory = m; return hipSuccess; }
inline hipError_t hipFree(void* p) { if (!rt().held.erase(p)) std::abort(); return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
'''

PROG = r'''
#include "device_pool.hpp"
#include <cstdio>
#include <new>
bool no_memory = false;
void* operator new(size_t n) {
    if (no_memory) throw std::bad_alloc();
    return std::malloc(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
using lvrhip::DevicePool;
using lvrhip::IdleScope;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
static DevicePool& pool() { return DevicePool::get(); }
static void* take(size_t n) { void* p = nullptr; if (pool().alloc(&p, n) != hipSuccess) std::abort(); return p; }
static void call(size_t n) { IdleScope s; void* p = take(n); s.set(); pool().free(p, IdleScope::flag()); }
int main(int argc, char** argv) {
    const size_t MB = 1 << 20;
    switch (argv[1][0]) {
        case 'k': {  // a block is kept and serves the next call of its size
            call(MB);
            CHECK(rt().held.size() == 1);
            void* p = rt().held.begin()->first;
            CHECK(take(MB) == p);
            pool().free(p, false);  // not known to be idle: back to the runtime
            CHECK(rt().held.empty());
            return 0;
        }
        case 'a': {  // host-array calls age what nobody takes, on every device
            rt().dev = 1;
            call(8 * MB);
            rt().dev = 0;
            call(16 * MB);
            for (int i = 0; i < 200; i++) call(1000);
            CHECK(rt().on(1) == 0);
            CHECK(rt().on(0) == 4096);
            return 0;
        }
        case 'r': {  // all of one device, then all
            for (int d = 0; d < 2; d++) {
                rt().dev = d;
                call(3 * MB);
                call(5 * MB);
            }
            void* live = take(7 * MB);
            CHECK(pool().release(0) == 8 * MB);
            CHECK(rt().on(0) == 0 && rt().on(1) == 15 * MB);
            CHECK(pool().release(DevicePool::ALL) == 8 * MB);
            CHECK(rt().on(1) == 7 * MB);
            CHECK(pool().release(DevicePool::ALL) == 0);
            pool().free(live, true);
            CHECK(pool().release(1) == 7 * MB && rt().held.empty());
            return 0;
        }
        case 'h': {  // no host memory: blocks go back to the runtime, and nothing throws where nothing may
            call(6 * MB);
            void* p = take(2 * MB);
            const size_t held = rt().held.size();
            no_memory = true;
            pool().free(p, true);
            CHECK(rt().held.size() == held - 1);
            pool().tick();
            uint32_t* w = nullptr;
            CHECK(pool().alloc_pinned(&w) == hipSuccess);
            pool().free_pinned(w, true);
            bool thrown = false;
            try {
                take(MB);
            } catch (const std::bad_alloc&) {
                thrown = true;
            }
            CHECK(thrown && rt().held.size() == held - 1);
            CHECK(pool().release(0) == 6 * MB);
            no_memory = false;
            CHECK(rt().held.empty());
            return 0;
        }
        case 'e': {  // what is too large to be kept is allocated as asked for, however large
            const size_t sizes[] = {512 * MB + 1, 700 * MB + 5, ~(size_t)0 - 7};
            for (size_t n : sizes) {
                void* p = take(n);
                CHECK(rt().held[p].second == n);
                pool().free(p, true);
                CHECK(rt().held.empty());
            }
            void* p = take(512 * MB - 1);
            CHECK(rt().held[p].second >= 512 * MB - 1 && rt().held[p].second <= 512 * MB);
            pool().free(p, true);
            CHECK(rt().held.size() == 1);
            return 0;
        }
        case 'b': {  // bounded
            for (int i = 0; i < 20; i++) {
                IdleScope s;
                std::vector<void*> v;
                for (int j = 0; j < 20; j++) v.push_back(take((200 + j) * MB));
                s.set();
                for (void* p : v) pool().free(p, IdleScope::flag());
            }
            CHECK(rt().on(0) <= DevicePool::CACHE_BYTES && rt().on(0) > 0);
            return 0;
        }
    }
    return 2;
}
'''


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "pool.cpp").write_text(PROG)
    r = subprocess.run(["g++", "-std=c++17", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", f"-I{d}",
                        "-I", os.path.join(ROOT, "lvr2_amd", "csrc"), str(d / "pool.cpp"), "-o", str(d / "pool"),
                        "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(d / "pool")


@pytest.mark.parametrize("what", ["kept", "aged", "released", "host memory", "exact", "bounded"])
def test_pool(exe, what):
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=60,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
