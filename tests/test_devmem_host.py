"""The cache of freed device blocks (csrc/devmem.hip) on the host, against a stand-in
for the runtime that knows which device still works and which calls a stream
capture forbids: a block is handed out again only after its own device was waited
for, the bound holds with the oldest blocks leaving first, and failed calls leave
no error behind."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "vk-rt-cuda-raytracing_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstddef>
#include <map>
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorStreamCaptureUnsupported = 900;
struct Runtime {
    int current = 0, error = 0;
    bool busy[2] = {false, false}, capture = false;
    size_t room = ~size_t(0), held = 0;
    std::map<void*, std::pair<size_t, int>> blocks;
    std::map<void*, int> freed;                     // order in which blocks were freed
    size_t next = 4096;
};
extern Runtime R;
inline hipError_t fail(hipError_t e) { R.error = e; return e; }
inline hipError_t hipGetDevice(int* d) { *d = R.current; return hipSuccess; }
inline hipError_t hipGetLastError() { const int e = R.error; R.error = 0; return e; }
inline hipError_t hipDeviceSynchronize() {
    if (R.capture) return fail(hipErrorStreamCaptureUnsupported);
    R.busy[R.current] = false;
    return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) {
    if (R.held + n > R.room) return fail(hipErrorOutOfMemory);
    *p = (void*)R.next;
    R.next += n + 4096;
    R.held += n;
    R.blocks[*p] = {n, R.current};
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    if (R.capture) return fail(hipErrorStreamCaptureUnsupported);
    auto it = R.blocks.find(p);
    if (it == R.blocks.end()) return fail(1);
    R.busy[it->second.second] = false;              // waits for the block's device
    R.held -= it->second.first;
    R.blocks.erase(it);
    const int k = (int)R.freed.size();
    R.freed[p] = k;
    return hipSuccess;
}
"""

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "hip/hip_runtime.h"
#include "rt_internal.h"
Runtime R;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
constexpr size_t MB = size_t(1) << 20, GB = size_t(1) << 30;

static void released_block_waits() {
    void* a = rt::dev_alloc(64 * MB);
    R.busy[0] = true;
    rt::dev_release(a);
    CHECK(rt::dev_alloc(64 * MB) == a && !R.busy[0]);
}
static void idle_block_does_not_wait() {
    void* a = rt::dev_alloc(64 * MB);
    rt::dev_free(a);
    R.busy[0] = true;
    CHECK(rt::dev_alloc(64 * MB) == a && R.busy[0]);
}
static void other_device() {
    R.current = 1;
    void* a = rt::dev_alloc(64 * MB);
    R.busy[1] = true;
    R.current = 0;                                  // destroyed while another device is current
    rt::dev_release(a);
    CHECK(rt::dev_alloc(64 * MB) != a);
    R.current = 1;
    CHECK(rt::dev_alloc(64 * MB) == a && !R.busy[1]);
}
static void release_after_the_wait() {
    void* a = rt::dev_alloc(64 * MB);
    void* b = rt::dev_alloc(256 * MB);
    rt::dev_release(a);
    CHECK(rt::dev_alloc(64 * MB) == a);             // waited here
    R.busy[0] = true;
    rt::dev_release(b);
    CHECK(rt::dev_alloc(256 * MB) == b && !R.busy[0]);
}
static void no_wait_possible() {
    void* a = rt::dev_alloc(64 * MB);
    R.busy[0] = true;
    R.capture = true;
    rt::dev_release(a);
    void* b = rt::dev_alloc(64 * MB);
    CHECK(b && b != a && R.busy[0]);
    CHECK(hipGetLastError() == 0);
    R.capture = false;
    CHECK(rt::dev_alloc(64 * MB) == a && !R.busy[0]);
}
static void bound_oldest_first() {
    std::vector<void*> p;
    for (int k = 0; k < 10; k++) p.push_back(rt::dev_alloc(256 * MB));
    for (void* x : p) rt::dev_free(x);
    CHECK(R.held == 2 * GB);
    CHECK(R.freed.size() == 2 && R.freed.at(p[0]) == 0 && R.freed.at(p[1]) == 1);
    void* big = rt::dev_alloc(3 * GB);
    rt::dev_free(big);                              // over the bound alone: the others stay
    CHECK(R.held == 2 * GB && R.freed.count(big));
    for (int k = 0; k < 8; k++) CHECK(rt::dev_alloc(256 * MB) != nullptr);
    CHECK(R.held == 2 * GB);                        // all eight served from the cache
    rt::dev_trim();
    CHECK(R.held == 2 * GB);                        // they are in use
}
static void bound_after_a_refused_free() {
    std::vector<void*> p;
    for (int k = 0; k < 10; k++) p.push_back(rt::dev_alloc(256 * MB));
    R.capture = true;
    for (void* x : p) rt::dev_free(x);
    CHECK(R.blocks.size() == 10 && hipGetLastError() == 0);   // none lost
    R.capture = false;
    void* q = rt::dev_alloc(16 * MB);
    rt::dev_free(q);
    CHECK(R.held <= 2 * GB);
    rt::dev_trim();
    CHECK(R.held == 0);
}
static void full_device() {
    void* a = rt::dev_alloc(64 * MB);
    rt::dev_free(a);
    R.room = 96 * MB;
    void* b = rt::dev_alloc(80 * MB);               // fails, gives the cache back, succeeds
    CHECK(b && R.held == 80 * MB && hipGetLastError() == 0);
    CHECK(!rt::dev_alloc(80 * MB) && hipGetLastError() == 0);
    rt::dev_release(b);
    void* c = rt::dev_alloc(1000);
    CHECK(c && R.held <= R.room);
    rt::dev_free(c);
    CHECK(R.freed.count(c));                        // small blocks are not kept
}
static void full_device_other_memory() {
    void* a = rt::dev_alloc(64 * MB);
    rt::dev_free(a);
    R.room = 96 * MB;
    int *p = nullptr, *q = (int*)1, *r = nullptr;
    CHECK(rt::dev_malloc(&p, 80 * MB) && p && R.held == 80 * MB);
    CHECK(!rt::dev_malloc(&q, 80 * MB) && !q && hipGetLastError() == 0);
    CHECK(rt::dev_malloc(&r, 0) && r);
}
int main(int, char** v) {
#define RUN(f) if (!strcmp(v[1], #f)) { f(); return 0; }
    RUN(released_block_waits) RUN(idle_block_does_not_wait) RUN(other_device) RUN(release_after_the_wait)
    RUN(no_wait_possible) RUN(bound_oldest_first) RUN(bound_after_a_refused_free) RUN(full_device)
    RUN(full_device_other_memory)
    return 2;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("devmem")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "driver.cpp").write_text(DRIVER)
    exe = str(d / "driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(d), "-I", CSRC,
                    "-x", "c++", os.path.join(CSRC, "devmem.hip"), str(d / "driver.cpp"), "-o", exe, "-lpthread"],
                   check=True)
    return exe


@pytest.mark.parametrize("case", ["released_block_waits", "idle_block_does_not_wait", "other_device",
                                  "release_after_the_wait", "no_wait_possible", "bound_oldest_first",
                                  "bound_after_a_refused_free", "full_device",
                                  "full_device_other_memory"])
def test_cache(driver, case):
    r = subprocess.run([driver, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
