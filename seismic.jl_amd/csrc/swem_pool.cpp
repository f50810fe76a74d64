// swem_pool.cpp -- device memory of the one-call entry points (swem_shots, swem_wem, swem_eshots,
// swem_compute_angles ...), which build a plan, run it and drop it.
//
// A call's blocks go back to a per-device list instead of hipFree, and the next call takes blocks that
// fit from it: the driver clears freed memory before it hands it out again, so a call that allocates
// its 10.5 GB of phase tables (the 1024 x 500 PSPI grid) anew waited up to 300 ms for a 12 ms march
// (339 -> 20 ms per call in a loop of calls).
//
// The list is bounded (kKeep per device and a share of the device's free memory, so that several processes
// on one device, each with its list, leave it room; least recently used blocks go first), drops blocks that
// the last few calls did not take, and is given back whole before a plan or a server is created, when
// an allocation of the library fails, so those see the memory a process without it would, and by
// swem_release_memory.  A block belongs to one call at a time; it returns to the list after the
// device has finished the call.
#include <algorithm>
#include <mutex>
#include <new>

#include "swem_plan.hpp"

namespace swem {

namespace {

constexpr size_t kKeep = size_t(16) << 30;  // bytes kept per device between calls, at most,
constexpr size_t kShare = 8;                // and of the free memory at the end of a call one part in this many
constexpr int kIdleCalls = 4;               // calls a block may stay unused
constexpr int kDevices = 64;

struct Block {
    void* p;
    size_t n;
    unsigned long long used;  // call that last held it
};

struct Pool {
    std::mutex mu;
    std::vector<Block> free;
    size_t kept = 0;
    unsigned long long calls = 0;

    void drop(size_t i)  // with mu held
    {
        (void)hipFree(free[i].p);
        kept -= free[i].n;
        free[i] = free.back();
        free.pop_back();
    }
};

bool has_pool(int dev) { return dev >= 0 && dev < kDevices; }

Pool& pool_of(int dev)  // of a device that has one
{
    static Pool* pools = new Pool[kDevices];  // never destroyed: the runtime may be gone at exit
    return pools[dev];
}

void trim(Pool& q)
{
    std::lock_guard<std::mutex> lock(q.mu);
    while (!q.free.empty()) q.drop(q.free.size() - 1);
}

}  // namespace

void trim_call_memory(int dev)
{
    if (has_pool(dev)) trim(pool_of(dev));
}

hipError_t device_malloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess) trim_call_memory(dev);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

CallMemory::CallMemory(int device) : dev(device)
{
    // inside a served request or another call, or no list for the device: plain allocations
    if (tl_dev_alloc || !has_pool(device)) return;
    tl_dev_alloc = this;
    on = true;
}

CallMemory::~CallMemory()
{
    if (!on) return;
    tl_dev_alloc = nullptr;
    if (blocks.empty()) return;
    (void)hipSetDevice(dev);
    (void)hipDeviceSynchronize();  // an early return may leave the call's work in flight
    Pool& q = pool_of(dev);
    std::lock_guard<std::mutex> lock(q.mu);
    const unsigned long long now = ++q.calls;
    try {
        q.free.reserve(q.free.size() + blocks.size());
    } catch (const std::bad_alloc&) {  // no room to note them: they go
        for (const Held& b : blocks) (void)hipFree(b.p);
        return;
    }
    for (const Held& b : blocks) {
        q.free.push_back({b.p, b.n, now});
        q.kept += b.n;
    }
    for (size_t i = q.free.size(); i-- > 0;)
        if (q.free[i].used + kIdleCalls < now) q.drop(i);
    size_t fr = 0, tot = 0, most = kKeep;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess) most = std::min(kKeep, (fr + q.kept) / kShare);
    while (q.kept > most) {
        size_t old = 0;  // the least recently used, the largest of them
        for (size_t i = 1; i < q.free.size(); i++)
            if (q.free[i].used < q.free[old].used || (q.free[i].used == q.free[old].used && q.free[i].n > q.free[old].n)) old = i;
        q.drop(old);
    }
}

void* CallMemory::alloc(size_t bytes)
{
    // a block the call has released again, or one of the list: the smallest that wastes at most a
    // quarter of it (small ones: up to 64 KiB)
    const size_t most = bytes + std::max(bytes / 3, size_t(64) << 10);
    Held* own = nullptr;
    for (Held& b : blocks)
        if (!b.taken && b.n >= bytes && b.n <= most && (!own || b.n < own->n)) own = &b;
    if (own) {
        own->taken = true;
        return own->p;
    }
    try {
        blocks.reserve(blocks.size() + 1);
    } catch (const std::bad_alloc&) {
        return nullptr;
    }
    Pool& q = pool_of(dev);
    void* p = nullptr;
    size_t n = 0;
    {
        std::lock_guard<std::mutex> lock(q.mu);
        size_t best = q.free.size();
        for (size_t i = 0; i < q.free.size(); i++)
            if (q.free[i].n >= bytes && q.free[i].n <= most && (best == q.free.size() || q.free[i].n < q.free[best].n)) best = i;
        if (best < q.free.size()) {
            p = q.free[best].p;
            n = q.free[best].n;
            q.kept -= n;
            q.free[best] = q.free.back();
            q.free.pop_back();
        }
    }
    if (!p) {
        n = (bytes + 255) & ~size_t(255);
        if (device_malloc(&p, n) != hipSuccess) return nullptr;
    }
    blocks.push_back({p, n, true});
    return p;
}

void CallMemory::release(void* p, size_t)
{
    for (Held& b : blocks)
        if (b.p == p) b.taken = false;
}

size_t CallMemory::spare() const
{
    Pool& q = pool_of(dev);
    std::lock_guard<std::mutex> lock(q.mu);
    return q.kept;
}

size_t device_free_bytes()
{
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) return 0;
    return fr + (tl_dev_alloc ? tl_dev_alloc->spare() : 0);
}

}  // namespace swem
