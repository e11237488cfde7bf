// Device block pool (dev_pool.hpp).
#include "dev_pool.hpp"

#include <algorithm>
#include <list>
#include <mutex>
#include <unordered_map>

#include "hip_util.hpp"

namespace cptc {

namespace {

struct Pool
{
    std::mutex mu;
    std::unordered_map<void*, PoolBlock> live;   // handed out by a scope
    std::list<PoolBlock> idle;                   // oldest first
    size_t idle_bytes = 0;
};

// never destroyed: at process exit the runtime may already be torn down
Pool& pool()
{
    static Pool* p = new Pool();
    return *p;
}

thread_local PoolScope* tl_scope = nullptr;

// a power of two up to 1 MiB, then multiples of 2 MiB (the device's page)
size_t round_up(size_t b)
{
    if (b <= (size_t(1) << 20))
    {
        size_t r = 512;
        while (r < b) r *= 2;
        return r;
    }
    const size_t m = size_t(2) << 20;
    return (b + m - 1) / m * m;
}

// whether a block of `have` bytes may stand for one of `need`
bool fits(size_t have, size_t need)
{
    return have >= need && have - need <= std::min(need / 2, POOL_WASTE_MAX);
}

// to the idle list; `out`: blocks that it pushes over the limit
void give(Pool& P, const PoolBlock& b, std::vector<PoolBlock>& out)
{
    if (b.bytes > POOL_IDLE_MAX)
    {
        out.push_back(b);
        return;
    }
    while (P.idle_bytes + b.bytes > POOL_IDLE_MAX)
    {
        out.push_back(P.idle.front());
        P.idle_bytes -= P.idle.front().bytes;
        P.idle.pop_front();
    }
    P.idle.push_back(b);
    P.idle_bytes += b.bytes;
}

void release(const std::vector<PoolBlock>& v)
{
    for (const PoolBlock& b : v) (void)hipFree(b.p);
}

// everything queued on device `dev` has finished
hipError_t device_wait(int dev)
{
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (cur != dev) (void)hipSetDevice(cur);
    return e;
}

}  // namespace

PoolScope::PoolScope(hipStream_t s, bool idle) : s_(s), idle_(idle), prev_(tl_scope)
{
    tl_scope = this;
}

PoolScope::~PoolScope()
{
    tl_scope = prev_;
    if (freed_.empty()) return;
    if (!idle_ && hipStreamSynchronize(s_) != hipSuccess)
    {
        release(freed_);   // hipFree waits by itself
        return;
    }
    std::vector<PoolBlock> out;
    {
        Pool& P = pool();
        std::lock_guard<std::mutex> lk(P.mu);
        for (const PoolBlock& b : freed_) give(P, b, out);
    }
    release(out);
}

hipError_t dev_malloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    pool_release();
    return hipMalloc(p, bytes);
}

int dev_alloc_bytes(void** p, size_t bytes)
{
    *p = nullptr;
    PoolScope* sc = tl_scope;
    if (!sc)
    {
        CPTC_HIP(dev_malloc(p, bytes));
        return CPTC_OK;
    }
    PoolBlock b;
    CPTC_HIP(hipGetDevice(&b.dev));
    const size_t need = round_up(bytes);
    // the smallest block that fits: the scope's own first, then an idle one
    size_t at = sc->freed_.size();
    for (size_t i = 0; i < sc->freed_.size(); ++i)
        if (sc->freed_[i].dev == b.dev && fits(sc->freed_[i].bytes, need) &&
            (at == sc->freed_.size() || sc->freed_[i].bytes < sc->freed_[at].bytes))
            at = i;
    Pool& P = pool();
    std::unique_lock<std::mutex> lk(P.mu);
    if (at < sc->freed_.size())
    {
        b = sc->freed_[at];
        sc->freed_[at] = sc->freed_.back();
        sc->freed_.pop_back();
        sc->freed_bytes_ -= b.bytes;
    }
    else
    {
        auto best = P.idle.end();
        for (auto it = P.idle.begin(); it != P.idle.end(); ++it)
            if (it->dev == b.dev && fits(it->bytes, need) &&
                (best == P.idle.end() || it->bytes < best->bytes))
                best = it;
        if (best != P.idle.end())
        {
            b = *best;
            P.idle_bytes -= b.bytes;
            P.idle.erase(best);
        }
    }
    if (!b.p)
    {
        lk.unlock();
        b.bytes = need;
        hipError_t e = dev_malloc(&b.p, need);
        if (e == hipErrorOutOfMemory && need > bytes && bytes > 0)
        {
            (void)hipGetLastError();
            b.bytes = bytes;
            e = hipMalloc(&b.p, bytes);
        }
        CPTC_HIP(e);
        lk.lock();
    }
    P.live[b.p] = b;
    *p = b.p;
    return CPTC_OK;
}

void dev_free(void* p)
{
    if (!p) return;
    Pool& P = pool();
    PoolBlock b;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        auto it = P.live.find(p);
        if (it != P.live.end())
        {
            b = it->second;
            P.live.erase(it);
        }
    }
    if (!b.p)   // not the pool's
        (void)hipFree(p);
    else if (PoolScope* sc = tl_scope)
    {
        if (sc->freed_bytes_ + b.bytes > POOL_SCOPE_MAX)
        {
            (void)hipFree(p);   // waits by itself
            return;
        }
        sc->freed_.push_back(b);
        sc->freed_bytes_ += b.bytes;
    }
    else if (device_wait(b.dev) != hipSuccess)   // hipFree's own wait
        (void)hipFree(p);
    else
    {
        std::vector<PoolBlock> out;
        {
            std::lock_guard<std::mutex> lk(P.mu);
            give(P, b, out);
        }
        release(out);
    }
}

void pool_trim()
{
    std::vector<PoolBlock> out;
    Pool& P = pool();
    {
        std::lock_guard<std::mutex> lk(P.mu);
        out.assign(P.idle.begin(), P.idle.end());
        P.idle.clear();
        P.idle_bytes = 0;
    }
    release(out);
}

void pool_release()
{
    for (PoolScope* sc = tl_scope; sc; sc = sc->prev_)
    {
        if (!sc->idle_ && !sc->freed_.empty()) (void)hipStreamSynchronize(sc->s_);
        release(sc->freed_);
        sc->freed_.clear();
        sc->freed_bytes_ = 0;
    }
    pool_trim();
}

}  // namespace cptc

extern "C" int cptc_dev_trim(void)
{
    cptc::pool_trim();
    return CPTC_OK;
}
