#pragma once
/*
 * The HIP calls of the host-side copies and allocations over a model of two
 * devices in host memory: what belongs to which device, which device is
 * current in a thread, and the calls that are refused for it.
 */
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>

enum hipError_t
{
    hipSuccess = 0,
    hipErrorInvalidValue = 1,
    hipErrorOutOfMemory = 2,
    hipErrorInvalidHandle = 400
};
enum
{
    hipMemcpyHostToDevice,
    hipMemcpyDeviceToHost,
    hipHostMallocDefault = 0,
    hipEventDisableTiming = 0,
    hipStreamNonBlocking = 1
};
using hipDevice_t = int;

struct StubStream
{
    int dev;
};
struct StubEvent
{
    int dev;
};
#define __device__
#define __host__
#define __global__

// Memory is counted, not given: a device holds STUB_CAP bytes, a pool keeps up
// to `keep` of what was freed to it.
constexpr uint64_t STUB_CAP = 16ull << 30;
struct StubPool
{
    int dev;
    uint64_t keep;
    uint64_t reserved;
    uint64_t used;
};
using hipStream_t = StubStream *;
using hipEvent_t = StubEvent *;
using hipMemPool_t = StubPool *;
enum hipMemPoolAttr
{
    hipMemPoolAttrReleaseThreshold
};
enum
{
    hipMemAllocationTypePinned = 1,
    hipMemLocationTypeDevice = 1
};
struct hipMemLocation
{
    int type;
    int id;
};
struct hipMemPoolProps
{
    int allocType;
    int handleTypes;
    hipMemLocation location;
    unsigned char reserved[64];
};

struct StubMemory
{
    std::mutex mu;
    uint64_t taken[2] = {0, 0}; // of each device, pools included
    StubPool def[2] = {{0, 0, 0, 0}, {1, 0, 0, 0}};
    std::map<void *, std::pair<StubPool *, uint64_t>> live;
    std::map<void *, std::pair<int, uint64_t>> plain;
    std::map<StubPool *, int> pools;
};
inline StubMemory & stub_memory()
{
    static StubMemory m;
    return m;
}

inline int & stub_current()
{
    static thread_local int d = 0;
    return d;
}

inline char const * hipGetErrorString(hipError_t) { return "refused"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int * d)
{
    *d = stub_current();
    return hipSuccess;
}
inline hipError_t hipSetDevice(int d)
{
    stub_current() = d;
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t * s, unsigned)
{
    *s = new StubStream{stub_current()};
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s)
{
    delete s;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t * d)
{
    *d = s->dev;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned)
{
    *e = new (std::nothrow) StubEvent{stub_current()};
    return *e != nullptr ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return e->dev == s->dev ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void ** p, size_t n, unsigned)
{
    *p = std::malloc(n);
    return *p != nullptr ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void * p)
{
    std::free(p);
    return hipSuccess;
}
inline std::atomic<int> & stub_copies()
{
    static std::atomic<int> n{0};
    return n;
}
inline hipError_t hipMemcpyAsync(void * d, void const * s, size_t n, int, hipStream_t)
{
    ++stub_copies();
    std::memcpy(d, s, n);
    return hipSuccess;
}

// The stream-ordered pools.  Only a synchronisation gives anything back.
inline hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t * p, int dev)
{
    *p = &stub_memory().def[dev];
    return hipSuccess;
}
inline hipError_t hipMemPoolCreate(hipMemPool_t * p, hipMemPoolProps const * q)
{
    *p = new StubPool{q->location.id, 0, 0, 0};
    return hipSuccess;
}
inline hipError_t hipMemPoolSetAttribute(hipMemPool_t p, hipMemPoolAttr, void * v)
{
    p->keep = *static_cast<uint64_t *>(v);
    return hipSuccess;
}
inline hipError_t hipMemPoolTrimTo(hipMemPool_t p, size_t keep)
{
    StubMemory & m = stub_memory();
    std::lock_guard<std::mutex> const lock(m.mu);
    uint64_t const want = p->used > keep ? p->used : keep;
    if (p->reserved > want)
    {
        m.taken[p->dev] -= p->reserved - want;
        p->reserved = want;
    }
    return hipSuccess;
}
inline hipError_t hipMallocFromPoolAsync(void ** ptr, size_t n, hipMemPool_t p, hipStream_t)
{
    StubMemory & m = stub_memory();
    std::lock_guard<std::mutex> const lock(m.mu);
    if (p->used + n > p->reserved)
    {
        uint64_t const more = p->used + n - p->reserved;
        if (m.taken[p->dev] + more > STUB_CAP)
        {
            return hipErrorOutOfMemory;
        }
        m.taken[p->dev] += more;
        p->reserved += more;
    }
    p->used += n;
    *ptr = std::malloc(1);
    m.live[*ptr] = {p, n};
    return hipSuccess;
}
inline hipError_t hipMallocAsync(void ** ptr, size_t n, hipStream_t s)
{
    return hipMallocFromPoolAsync(ptr, n, &stub_memory().def[s->dev], s);
}
inline hipError_t hipFreeAsync(void * ptr, hipStream_t)
{
    StubMemory & m = stub_memory();
    std::lock_guard<std::mutex> const lock(m.mu);
    auto const it = m.live.find(ptr);
    it->second.first->used -= it->second.second;
    m.live.erase(it);
    std::free(ptr);
    return hipSuccess;
}
template <typename T>
hipError_t hipMalloc(T ** ptr, size_t n)
{
    StubMemory & m = stub_memory();
    std::lock_guard<std::mutex> const lock(m.mu);
    int const d = stub_current();
    if (m.taken[d] + n > STUB_CAP)
    {
        return hipErrorOutOfMemory;
    }
    m.taken[d] += n;
    *ptr = static_cast<T *>(std::malloc(1));
    m.plain[*ptr] = {d, n};
    return hipSuccess;
}
inline hipError_t hipFree(void * ptr)
{
    StubMemory & m = stub_memory();
    std::lock_guard<std::mutex> const lock(m.mu);
    auto const it = m.plain.find(ptr);
    m.taken[it->second.first] -= it->second.second;
    m.plain.erase(it);
    std::free(ptr);
    return hipSuccess;
}
