"""The device block pool (host/dev_pool.cpp) on a device that is only counted:
the pool and the runtime helpers are compiled here against a handful of HIP
functions that keep a byte budget per device, so that the paths taken when the
device has no room can be walked through without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "cptc_amd", "csrc", "host")

SOURCE = r'''
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "dev_pool.hpp"
#include "hip_util.hpp"

// ---- the counted devices
static size_t used[2], peak[2], limit[2];
static int cur, waits[2], stream_waits;
static std::map<void*, std::pair<int, size_t>> blocks;
static uintptr_t next_p = 1 << 20;

extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (n == 0) return hipSuccess;
    if (used[cur] + n > limit[cur]) return hipErrorOutOfMemory;
    used[cur] += n;
    if (used[cur] > peak[cur]) peak[cur] = used[cur];
    *p = reinterpret_cast<void*>(next_p);
    next_p += 4096;
    blocks[*p] = {cur, n};
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end())
    {
        std::printf("a block freed twice\n");
        std::exit(1);
    }
    ++waits[it->second.first];   // hipFree waits for its device
    used[it->second.first] -= it->second.second;
    blocks.erase(it);
    return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int* d) { *d = cur; return hipSuccess; }
extern "C" hipError_t hipSetDevice(int d) { cur = d; return hipSuccess; }
extern "C" hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { ++stream_waits; return hipSuccess; }
extern "C" hipError_t hipDeviceSynchronize() { ++waits[cur]; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" const char* hipGetErrorString(hipError_t) { return "error"; }
extern "C" hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
extern "C" hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }

#define CHECK(c)                                                        \
    do                                                                  \
    {                                                                   \
        if (!(c))                                                       \
        {                                                               \
            std::printf("line %d: %s (%s)\n", __LINE__, #c, cptc_last_error()); \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

using namespace cptc;
static const size_t MiB = size_t(1) << 20, GiB = size_t(1) << 30;
static hipStream_t S = reinterpret_cast<hipStream_t>(8);

static void reset(size_t lim)
{
    pool_trim();
    CHECK(used[0] == 0 && used[1] == 0);
    cur = 0;
    for (int d = 0; d < 2; ++d) peak[d] = 0, waits[d] = 0, limit[d] = lim;
    stream_waits = 0;
}

// A set-up's allocations and frees, drawn; what it still holds at the end is
// left in `kept`.  0 when an allocation failed.
static int setup(unsigned seed, bool pooled, std::vector<void*>& kept, size_t* excess)
{
    unsigned x = seed * 2654435761u + 12345u;
    auto rnd = [&](unsigned n) { x = x * 1664525u + 1013904223u; return (x >> 8) % n; };
    std::vector<std::pair<void*, size_t>> live;
    *excess = 0;
    int ok = 1;
    auto get = [&](size_t n) {
        void* p = nullptr;
        if (pooled ? dev_alloc_bytes(&p, n) != CPTC_OK : hipMalloc(&p, n) != hipSuccess) ok = 0;
        else live.push_back({p, n});
    };
    auto put = [&](size_t i) {
        if (pooled) dev_free(live[i].first);
        else (void)hipFree(live[i].first);
        live.erase(live.begin() + long(i));
    };
    for (int step = 0; step < 60 && ok; ++step)
    {
        get(rnd(4) == 0 ? size_t(rnd(3000000)) + 1 : size_t(rnd(600) + 1) * MiB + rnd(1000));
        // a sort's scratch: larger each time, so that no freed block serves
        if (ok && step % 7 == 0)
        {
            get(size_t(200 + 90 * step) * MiB);
            if (ok) put(live.size() - 1);
        }
        if (ok && live.size() > 12) put(rnd(unsigned(live.size())));
    }
    for (auto& b : live)
    {
        kept.push_back(b.first);
        *excess += blocks[b.first].second - b.second;
    }
    return ok;
}

// What fits without the pool fits with it, up to the excess of the live blocks.
static void setups()
{
    for (unsigned seed = 1; seed <= 40; ++seed)
    {
        std::vector<void*> kept;
        size_t excess = 0;
        reset(1000 * GiB);
        CHECK(setup(seed, false, kept, &excess));
        const size_t plain = peak[0];
        for (void* p : kept) (void)hipFree(p);
        kept.clear();
        reset(1000 * GiB);
        {   // another handle's blocks lie idle
            PoolScope sc(S);
            CHECK(setup(seed + 100, true, kept, &excess));
            for (void* p : kept) dev_free(p);
            kept.clear();
        }
        CHECK(used[0] <= POOL_IDLE_MAX);
        // 13 live blocks and a scratch block at most
        limit[0] = plain + 14 * POOL_WASTE_MAX;
        {
            PoolScope sc(S);
            CHECK(setup(seed, true, kept, &excess));
            CHECK(excess <= kept.size() * POOL_WASTE_MAX);
        }
        {
            PoolScope sc(nullptr, true);
            for (void* p : kept) dev_free(p);
        }
        CHECK(used[0] <= POOL_IDLE_MAX);
    }
}

// An allocation that has room only at the size asked for
static void unrounded()
{
    reset(64 * MiB);
    limit[0] = 5 * MiB;
    void* p = nullptr;
    {
        PoolScope sc(S);
        CHECK(dev_alloc_bytes(&p, 5 * MiB) == CPTC_OK);
        dev_free(p);
        CHECK(dev_alloc_bytes(&p, 5 * MiB) == CPTC_OK);   // the 5 MiB go back for it
        dev_free(p);
        CHECK(dev_alloc_bytes(&p, 6 * MiB) != CPTC_OK && p == nullptr);
    }
}

// Idle blocks make room for every other allocation of the library
static void others()
{
    for (int which = 0; which < 4; ++which)
    {
        reset(1536 * MiB);
        std::vector<void*> v(9, nullptr);
        {
            PoolScope sc(S);
            for (void*& p : v) CHECK(dev_alloc_bytes(&p, 100 * MiB) == CPTC_OK);
            for (void* p : v) dev_free(p);
        }
        CHECK(used[0] == 900 * MiB);
        void* p = nullptr;
        if (which == 0) CHECK(dev_alloc_bytes(&p, 1400 * MiB) == CPTC_OK);
        if (which == 1) CHECK(cptc_dev_malloc(1400 * MiB, &p) == CPTC_OK);
        if (which == 2) CHECK(scratch_get(SCR_LAYOUT_A, 1400 * MiB, &p) == CPTC_OK);
        if (which == 3)
        {
            PoolScope sc(S);
            CHECK(dev_alloc_bytes(&p, 1400 * MiB) == CPTC_OK);
            dev_free(p);
            p = nullptr;
            CHECK(used[0] == 1400 * MiB);
        }
        if (which < 2) CHECK(cptc_dev_free(p) == CPTC_OK);
        if (which == 2)   // the scratch buffer stays: hand its bytes back here
        {
            used[0] -= blocks[p].second;
            blocks[p].second = 0;
        }
        else
            CHECK(used[0] == 0);
    }
}

// What a scope holds back is bounded
static void scope_bound()
{
    reset(1000 * GiB);
    {
        PoolScope sc(S);
        for (int i = 0; i < 20; ++i)
        {
            void* p = nullptr;
            CHECK(dev_alloc_bytes(&p, size_t(200 + 150 * i) * MiB) == CPTC_OK);
            dev_free(p);
            CHECK(used[0] <= POOL_SCOPE_MAX);
        }
    }
    CHECK(used[0] <= POOL_IDLE_MAX);
}

// A block freed outside a scope: its own device is waited for, the caller's
// current device stays; a scope's blocks wait for its stream
static void devices()
{
    reset(GiB);
    void* p = nullptr;
    cur = 1;
    {
        PoolScope sc(S);
        CHECK(dev_alloc_bytes(&p, MiB) == CPTC_OK);
    }
    cur = 0;
    waits[0] = waits[1] = 0;
    dev_free(p);
    CHECK(waits[1] == 1 && waits[0] == 0 && cur == 0);
    CHECK(used[1] == MiB);
    void* q = nullptr;
    {
        PoolScope sc(S);
        CHECK(dev_alloc_bytes(&q, MiB) == CPTC_OK);   // device 0: not that block
        CHECK(q != p && used[0] == MiB);
        dev_free(q);
        CHECK(stream_waits == 0);
    }
    CHECK(stream_waits == 1);
}

int main()
{
    setups();
    unrounded();
    others();
    scope_bound();
    devices();
    reset(GiB);
    std::printf("ok\n");
    std::fflush(stdout);
    std::_Exit(0);   // the scratch table outlives the counted device otherwise
}
'''


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    src, out = d / "pool.cpp", d / "pool"
    src.write_text(SOURCE)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-Wall",
                        "-Wno-unknown-pragmas", "-I", os.path.join(ROOT, "include"), "-I", HOST,
                        "-I", "/opt/rocm/include", str(src), os.path.join(HOST, "dev_pool.cpp"),
                        os.path.join(HOST, "runtime.cpp"), "-o", str(out), "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return str(out)


def test_pool_makes_room(exe):
    """A set-up that fits without the pool fits with it; idle blocks give way
    to the library's other allocations; what scopes hold back is bounded; a
    block's own device is waited for."""
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
