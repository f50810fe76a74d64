// Device memory of plans and one-call entry points (swem_plan.hpp, swem_pool.cpp) over a device made of
// counters: hipMalloc hands out host addresses against a set capacity.  One scenario per run
// (test_call_memory.py); exit status 0 where it holds.
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>

#include "swem_plan.hpp"

static long g_new_left = -1;  // host allocations until one fails (-1: none does)

// ------------------------------------------------------------------ the device
static size_t g_capacity = size_t(288) << 30, g_used = 0, g_mallocs = 0, g_syncs = 0;
static int g_device = 0;
static std::map<void*, std::pair<size_t, int>> g_live;  // bytes and device

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    g_mallocs++;
    if (g_used + n > g_capacity) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    const long left = g_new_left;  // (not of the library)
    g_new_left = -1;
    g_live[*p] = {n, g_device};
    g_new_left = left;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    auto it = g_live.find(p);
    if (it == g_live.end()) std::abort();
    g_used -= it->second.first;
    g_live.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = g_device, hipSuccess; }
hipError_t hipSetDevice(int d) { return g_device = d, hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return g_syncs++, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* fr, size_t* tot) { return *fr = g_capacity - g_used, *tot = g_capacity, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "device error"; }
}

// ------------------------------------------------------------------ the host: allocations that fail on demand
void* operator new(size_t n)
{
    if (g_new_left == 0) throw std::bad_alloc();
    if (g_new_left > 0) g_new_left--;
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace swem {
thread_local DevAllocator* tl_dev_alloc = nullptr;
thread_local HostStager* tl_stager = nullptr;
int set_error(int code, const char*, ...) { return code; }
int hip_error(hipError_t e, const char*, const char*, int) { return e == hipErrorOutOfMemory ? SWEM_ENOMEM : SWEM_EDEVICE; }
int upload_bytes(void*, const void*, size_t) { return SWEM_OK; }
}  // namespace swem

using namespace swem;
constexpr size_t GiB = size_t(1) << 30, MiB = size_t(1) << 20;

#define EXPECT(x)                                                             \
    do {                                                                      \
        if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1;       \
    } while (0)

// a call that takes the given sizes at once
template <class... S>
static int call(int device, S... bytes)
{
    return one_call(device, [&] {
        DevBuf<char> b[sizeof...(bytes)];
        const size_t n[] = {(size_t)bytes...};
        for (size_t i = 0; i < sizeof...(bytes); i++) SWEM_TRY(b[i].alloc(n[i]));
        return SWEM_OK;
    });
}

static int reuse()
{
    EXPECT(call(0, 3 * GiB, 70 * MiB) == SWEM_OK);
    const size_t first = g_mallocs;
    EXPECT(call(0, 3 * GiB - 5, 70 * MiB) == SWEM_OK && g_mallocs == first);  // the same blocks
    EXPECT(call(0, GiB) == SWEM_OK && g_mallocs == first + 1);                // not a block three times as large
    EXPECT(g_used == 4 * GiB + 70 * MiB && g_syncs == 3);
    return 0;
}

static int bounds()
{
    EXPECT(call(0, 9 * GiB, 9 * GiB) == SWEM_OK && g_used == 9 * GiB);  // at most 16 GiB stay
    for (int i = 0; i < 4; i++) EXPECT(call(0, 2 * GiB) == SWEM_OK && g_used == 11 * GiB);
    EXPECT(call(0, 2 * GiB) == SWEM_OK && g_used == 2 * GiB);  // unused by the last four calls
    // other processes have taken the rest: an eighth of what is left
    g_capacity = 40 * GiB;
    EXPECT(call(0, 4 * GiB, 2 * GiB) == SWEM_OK && g_used == 2 * GiB);
    EXPECT(call(0, 4 * GiB) == SWEM_OK && g_used == 4 * GiB);
    g_capacity = 10 * GiB;
    EXPECT(call(0, 2 * GiB) == SWEM_OK && g_used == 0);
    return 0;
}

static int given_back()
{
    EXPECT(call(0, 5 * GiB) == SWEM_OK && g_used == 5 * GiB);
    EXPECT(call(1, 3 * GiB) == SWEM_OK && g_used == 8 * GiB);
    trim_call_memory(0);
    EXPECT(g_used == 3 * GiB);
    trim_call_memory(1);
    EXPECT(g_used == 0 && g_live.empty());
    return 0;
}

// a resident plan's buffers grow after a call has filled the list
static int growth_after_call()
{
    DevBuf<char> table, work;
    EXPECT(table.alloc(4 * GiB) == SWEM_OK);
    EXPECT(call(0, 8 * GiB, 6 * GiB) == SWEM_OK && g_used == 18 * GiB);
    g_capacity = 20 * GiB;  // others took the rest
    EXPECT(work.alloc(12 * GiB) == SWEM_OK && g_used == 16 * GiB);
    void* p = nullptr;
    EXPECT(device_malloc(&p, 5 * GiB) == hipErrorOutOfMemory && !p);  // not there at all
    return 0;
}

// a call near the limit gets what plain allocations would give it: blocks that it released itself, and
// what kept blocks are larger than it asked for
static int call_at_the_limit()
{
    g_capacity = 20 * GiB;
    const int rc = one_call(0, [&] {
        DevBuf<char> a, b;
        SWEM_TRY(a.alloc(12 * GiB));
        a.release();
        return b.alloc(15 * GiB);
    });
    EXPECT(rc == SWEM_OK);
    trim_call_memory(0);
    g_capacity = 288 * GiB;
    EXPECT(call(0, 8 * GiB, 8 * GiB) == SWEM_OK);
    g_capacity = 20 * GiB;
    EXPECT(call(0, 6 * GiB + 1, 6 * GiB + 1, 7 * GiB) == SWEM_OK);
    EXPECT(call(0, 21 * GiB) == SWEM_ENOMEM);
    return 0;
}

static int buffers_free_themselves()
{
    {
        DevBuf<char> a, b;
        EXPECT(a.alloc(MiB) == SWEM_OK && b.alloc(2 * MiB) == SWEM_OK && g_used == 3 * MiB);
        DevBuf<char> c(std::move(a));
        EXPECT(!a.p && c.p && c.n == MiB);
        b = std::move(c);
        EXPECT(g_used == MiB && b.n == MiB && !c.p);
    }
    EXPECT(g_used == 0 && g_live.empty());
    return 0;
}

// no exception leaves the entry points, wherever the host runs out of memory
static int host_memory()
{
    EXPECT(call(0, MiB, 2 * MiB) == SWEM_OK);
    for (long left = 0; left < 12; left++) {
        g_new_left = left;
        const int rc = call(0, MiB, 2 * MiB, (3 + left) * MiB);
        g_new_left = -1;
        EXPECT(rc == SWEM_OK || rc == SWEM_ENOMEM);
        EXPECT(!tl_dev_alloc);
    }
    trim_call_memory(0);
    EXPECT(g_used == 0 && g_live.empty());
    return 0;
}

// a block belongs to the device it was taken on
static int many_devices()
{
    for (int d : {0, 63, 64, 200}) {
        g_device = d;
        EXPECT(call(d, MiB) == SWEM_OK);
    }
    for (int d : {0, 63, 64, 200}) {
        g_device = d;
        const int rc = one_call(d, [&] {
            DevBuf<char> b;
            SWEM_TRY(b.alloc(MiB));
            return g_live[b.p].second == d ? SWEM_OK : SWEM_EDEVICE;
        });
        EXPECT(rc == SWEM_OK);
    }
    return 0;
}

int main(int, char** argv)
{
    const std::map<std::string, int (*)()> all = {
        {"reuse", reuse}, {"bounds", bounds}, {"given_back", given_back},
        {"growth_after_call", growth_after_call}, {"call_at_the_limit", call_at_the_limit},
        {"buffers_free_themselves", buffers_free_themselves}, {"host_memory", host_memory},
        {"many_devices", many_devices}};
    return all.at(argv[1])();
}
