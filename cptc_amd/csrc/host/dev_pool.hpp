// Device blocks of a handle's set-up, reused from one allocation and one
// handle to the next.
//
// A set-up makes ~90 device allocations (sort scratch, views, tiles) and frees
// them with the handle; hipMalloc and hipFree of a few MB take 0.3 ms each
// (the pages are mapped and unmapped, and hipFree waits for the device):
// 11.6 of the 19.5 ms that a 1 M-nonzero order-3 job (set-up, 5 iterations,
// factors out) took; with the blocks kept and the initial factors drawn on a
// thread beside the set-up it takes 5.3 (with max_u32 in place of an OpenMP loop).
//
// dev_alloc / dev_free are hipMalloc / hipFree outside a PoolScope.  Inside
// one (on the thread that opened it), a block freed goes to the scope and may
// be handed out again in it at once: everything in a scope runs on the
// scope's one stream, so the next user's work is queued behind the last
// one's.  When the scope ends, its stream is waited for and the blocks become
// idle blocks of the process, which any scope may take.
//
// What the blocks cost in memory: idle ones are at most POOL_IDLE_MAX bytes
// (the oldest go back to the device first), a scope's freed ones at most
// POOL_SCOPE_MAX, and a block handed out is at most half as much again and
// POOL_WASTE_MAX larger than the rounded size asked for.  Every device allocation of the
// library goes through dev_malloc or dev_alloc: where the device has no room,
// the freed blocks of the thread's scopes and all idle ones go back to it and
// the allocation is tried again (in a scope, then at its unrounded size), so a
// set-up fails only if it would without the pool, up to that excess of its
// live blocks.  cptc_dev_trim returns the idle blocks on request.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <vector>

namespace cptc {

constexpr size_t POOL_IDLE_MAX = size_t(1) << 30;
constexpr size_t POOL_SCOPE_MAX = size_t(4) << 30;
constexpr size_t POOL_WASTE_MAX = size_t(8) << 20;

struct PoolBlock
{
    void* p = nullptr;
    size_t bytes = 0;
    int dev = 0;
};

class PoolScope
{
public:
    // Work on blocks freed in this scope is queued on `s`; with idle = true it
    // has all finished (s is not used).
    explicit PoolScope(hipStream_t s, bool idle = false);
    ~PoolScope();
    PoolScope(const PoolScope&) = delete;
    PoolScope& operator=(const PoolScope&) = delete;

private:
    friend int dev_alloc_bytes(void** p, size_t bytes);
    friend void dev_free(void* p);
    friend void pool_release();
    hipStream_t s_;
    bool idle_;
    PoolScope* prev_;
    std::vector<PoolBlock> freed_;
    size_t freed_bytes_ = 0;
};

// hipMalloc, once more after pool_release() where the device has no room
hipError_t dev_malloc(void** p, size_t bytes);
int dev_alloc_bytes(void** p, size_t bytes);
void dev_free(void* p);
void pool_trim();      // idle blocks of every device back to it
void pool_release();   // and the freed ones of this thread's scopes

template <class T>
int dev_alloc(T** p, size_t bytes)
{
    void* q = nullptr;
    const int rc = dev_alloc_bytes(&q, bytes);
    *p = static_cast<T*>(q);
    return rc;
}

}  // namespace cptc
