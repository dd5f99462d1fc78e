"""Device memory that contexts keep between calls (boostfractor.jl_amd/csrc/bf_pool.h) on the
CPU, on a runtime of 1000 blocks of memory that the test provides: an allocation that fails
for what any context of the device keeps is served, the limit holds and gives memory back,
blocks of plans that outlive their context are freed, and threads free what others keep."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "boostfractor.jl_amd", "csrc")

MAIN = r'''
#include "bf_pool.h"
#include <cstdio>
#include <cstdlib>
#include <thread>
constexpr size_t MB = (size_t)1 << 20, ROOM = 1000 * MB;
static std::mutex mu;
static std::map<void*, size_t> live[2];
static size_t used[2];
static thread_local int dev = 0;
static uintptr_t next = 4096;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lk(mu);
    if (used[dev] + n > ROOM) return hipErrorOutOfMemory;
    *p = (void*)(next += 4096);
    live[dev][*p] = n;
    used[dev] += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    for (int d = 0; d < 2; d++) {
        auto it = live[d].find(p);
        if (it == live[d].end()) continue;
        used[d] -= it->second;
        live[d].erase(it);
        return hipSuccess;
    }
    std::abort();
}
hipError_t hipGetDevice(int* d) { *d = dev; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
static thread_local std::shared_ptr<bf::DevPool> cur;
namespace bf { const std::shared_ptr<DevPool>& call_pool() { return cur; } }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    using bf::DevBuf;
    using bf::DevPool;
    auto a = std::make_shared<DevPool>(0), b = std::make_shared<DevPool>(0), c = std::make_shared<DevPool>(1);
    dev = 1;
    cur = c;
    { DevBuf x(600 * MB); }
    CHECK(used[1] == DevPool::round(600 * MB));
    dev = 0;
    cur = a;
    { DevBuf x(400 * MB), y(200 * MB); }
    CHECK(used[0] >= 600 * MB);  // kept
    { DevBuf x(400 * MB); CHECK(used[0] <= 660 * MB); }  // and taken again
    cur = b;
    { DevBuf x(900 * MB); CHECK(used[0] == 900 * MB); }  // what the other context kept, without the rounding
    CHECK(used[1] >= 600 * MB);  // not another device's
    b->trim();
    { DevBuf x(990 * MB); CHECK(used[0] == 990 * MB); }
    b->trim();
    bool refused = false;
    try { DevBuf x(1001 * MB); } catch (const bf::Error& e) { refused = e.code == BF_ERR_NOMEM; }
    CHECK(refused && used[0] == 0);
    cur = a;
    a->limit(100 * MB);
    { DevBuf x(64 * MB), y(32 * MB), z(32 * MB), w(256 * MB); }
    CHECK(used[0] <= 100 * MB && used[0] > 0);
    a->limit(0);
    CHECK(used[0] == 0);
    { DevBuf x(64 * MB); }
    CHECK(used[0] == 0);
    a->limit(DevPool::KEEP);
    {
        DevBuf plan(64 * MB);
        a->trim(true);  // the context is destroyed
        a.reset();
        cur.reset();
        CHECK(used[0] >= 64 * MB);
    }
    CHECK(used[0] == 0);
    dev = 0;
    std::vector<std::thread> ts;
    bool bad[4] = {};
    for (int t = 0; t < 4; t++)
        ts.emplace_back([t, &bad] {
            for (int k = 0; k < 200; k++) {
                cur = std::make_shared<DevPool>(0);
                try {
                    for (int q = 0; q < 5; q++) { DevBuf x((size_t)(50 + 10 * q + t) * MB), y(20 * MB); }
                } catch (const bf::Error&) { bad[t] = true; }
            }
            cur.reset();
        });
    for (auto& t : ts) t.join();
    for (bool v : bad) CHECK(!v);
    CHECK(used[0] == 0);
    std::printf("ok\n");
    return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_pool_of_freed_blocks(tmp_path):
    src = tmp_path / "pool.cpp"
    src.write_text(MAIN)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
