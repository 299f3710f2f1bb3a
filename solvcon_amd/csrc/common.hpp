#pragma once
/*
 * Shared plumbing of the HIP library: status codes and the thread-local
 * error message of the C ABI, HIP error checks, and launch helpers.
 *
 * Status codes map to the exception types the reference raises through
 * pybind11 (cpp/solvcon/multidim/pymod/wrap_multidim.cpp:42-67):
 *   SC_OK 0, SC_EVALUE 1 (ValueError), SC_EINDEX 2 (IndexError),
 *   SC_ERUNTIME 3 (RuntimeError), SC_EDEVICE 4 (a HIP failure).
 */

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <stdexcept>
#include <string>

namespace scamd
{

enum Status : int
{
    SC_OK = 0,
    SC_EVALUE = 1,
    SC_EINDEX = 2,
    SC_ERUNTIME = 3,
    SC_EDEVICE = 4,
};

struct Error : std::runtime_error
{
    int code;
    Error(int c, std::string const & m)
        : std::runtime_error(m)
        , code(c)
    {
    }
};

void set_last_error(int code, std::string const & msg);

[[noreturn]] inline void fail(int code, std::string const & msg) { throw Error(code, msg); }

inline void hip_check(hipError_t e, char const * what)
{
    if (e != hipSuccess)
    {
        fail(SC_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
    }
}

#define SC_HIP(call) ::scamd::hip_check((call), #call)

// Run f and turn exceptions into a status code plus the last-error message.
template <typename F>
int guard(F && f)
{
    try
    {
        f();
        return SC_OK;
    }
    catch (Error const & e)
    {
        set_last_error(e.code, e.what());
        return e.code;
    }
    catch (std::bad_alloc const &)
    {
        set_last_error(SC_ERUNTIME, "host allocation failed");
        return SC_ERUNTIME;
    }
    catch (std::exception const & e)
    {
        set_last_error(SC_ERUNTIME, e.what());
        return SC_ERUNTIME;
    }
}

// The stream that device allocations of the calling thread are ordered on:
// a handle sets it (AllocScope) while it works, so its buffers come from
// the stream-ordered pool (hipMallocAsync / hipFreeAsync) and freeing one
// never waits for the work of other handles' streams, as hipFree would.
inline hipStream_t & alloc_stream()
{
    static thread_local hipStream_t s = nullptr;
    return s;
}

struct AllocScope
{
    hipStream_t prev;
    explicit AllocScope(hipStream_t s)
        : prev(alloc_stream())
    {
        alloc_stream() = s;
    }
    ~AllocScope() { alloc_stream() = prev; }
    AllocScope(AllocScope const &) = delete;
    AllocScope & operator=(AllocScope const &) = delete;
};

// Makes a stream's device the current one for a while: events, streams and
// pinned buffers are made on the current device, which the caller may have
// changed since the handle was made, and an event is refused on a stream of
// another device.
struct OnDevice
{
    int dev = 0;
    int prev = 0;
    explicit OnDevice(hipStream_t s)
    {
        hipDevice_t d = 0;
        SC_HIP(hipStreamGetDevice(s, &d));
        SC_HIP(hipGetDevice(&prev));
        dev = static_cast<int>(d);
        if (dev != prev)
        {
            SC_HIP(hipSetDevice(dev));
        }
    }
    ~OnDevice()
    {
        if (dev != prev)
        {
            (void)hipSetDevice(prev);
        }
    }
    OnDevice(OnDevice const &) = delete;
    OnDevice & operator=(OnDevice const &) = delete;
};

// The library's own stream-ordered pool of each device, and how much it keeps
// for the next allocation instead of returning it to the system at every
// synchronisation.  Every table that is read back or loaded goes through a
// staging buffer, and every mesh build through a dozen scratch buffers:
// mapping them anew took a third of the set-up of a 131072-triangle solve
// (20.7 to 15.3 ms) and of a 156800-cell block's (29.8 to 19.4 ms).  A pool
// gives back whatever exceeds this at a synchronisation, and all that is free
// when an allocation of the library fails and when its last stream goes
// (StreamHolder).  The device's default pool is left as the application has it.
constexpr uint64_t POOL_KEEP = 4ull << 30;
constexpr int POOL_DEVICES = 64;

inline std::atomic<hipMemPool_t> & pool_slot(int dev)
{
    static std::atomic<hipMemPool_t> slots[POOL_DEVICES] = {};
    if (dev < 0 || dev >= POOL_DEVICES)
    {
        fail(SC_EDEVICE, "device index out of range");
    }
    return slots[dev];
}

// Never destroyed: the process's end takes it.
inline hipMemPool_t pool_of(int dev)
{
    std::atomic<hipMemPool_t> & slot = pool_slot(dev);
    hipMemPool_t pool = slot.load(std::memory_order_acquire);
    if (pool == nullptr)
    {
        static std::mutex mu;
        std::lock_guard<std::mutex> const lock(mu);
        pool = slot.load(std::memory_order_acquire);
        if (pool == nullptr)
        {
            hipMemPoolProps props{};
            props.allocType = hipMemAllocationTypePinned;
            props.location.type = hipMemLocationTypeDevice;
            props.location.id = dev;
            uint64_t keep = POOL_KEEP;
            SC_HIP(hipMemPoolCreate(&pool, &props));
            SC_HIP(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
            slot.store(pool, std::memory_order_release);
        }
    }
    return pool;
}

// Gives back what is free in the current device's pool, after all its work.
inline void pool_give_back()
{
    int dev = 0;
    SC_HIP(hipGetDevice(&dev));
    if (hipMemPool_t const pool = pool_slot(dev).load(std::memory_order_acquire))
    {
        SC_HIP(hipDeviceSynchronize());
        SC_HIP(hipMemPoolTrimTo(pool, 0));
    }
}

// hipMallocFromPoolAsync on the stream's device (hipMalloc on the current one
// without a stream), once more with the pool emptied when memory is short.
inline void pool_malloc(void ** ptr, size_t nb, hipStream_t s)
{
    auto const get = [&](int dev)
    { return s != nullptr ? hipMallocFromPoolAsync(ptr, nb, pool_of(dev), s) : hipMalloc(ptr, nb); };
    int dev = 0;
    if (s != nullptr)
    {
        hipDevice_t d = 0;
        SC_HIP(hipStreamGetDevice(s, &d));
        dev = static_cast<int>(d);
    }
    hipError_t e = get(dev);
    if (e == hipErrorOutOfMemory)
    {
        (void)hipGetLastError();
        if (s != nullptr)
        {
            OnDevice const on(s);
            pool_give_back();
        }
        else
        {
            pool_give_back();
        }
        e = get(dev);
    }
    SC_HIP(e);
}

// Device buffer owned by a handle; freed on the stream it was allocated on
// (or with hipFree when it was allocated outside any AllocScope).
template <typename T>
struct DevBuf
{
    T * ptr = nullptr;
    int64_t count = 0;
    hipStream_t stream = nullptr;

    DevBuf() = default;
    DevBuf(DevBuf const &) = delete;
    DevBuf & operator=(DevBuf const &) = delete;
    DevBuf(DevBuf && o) noexcept
        : ptr(o.ptr)
        , count(o.count)
        , stream(o.stream)
    {
        o.ptr = nullptr;
        o.count = 0;
        o.stream = nullptr;
    }
    DevBuf & operator=(DevBuf && o) noexcept
    {
        if (this != &o)
        {
            release();
            ptr = o.ptr;
            count = o.count;
            stream = o.stream;
            o.ptr = nullptr;
            o.count = 0;
            o.stream = nullptr;
        }
        return *this;
    }
    ~DevBuf() { release(); }

    void alloc(int64_t n)
    {
        release();
        if (n > 0)
        {
            stream = alloc_stream();
            size_t const nb = sizeof(T) * static_cast<size_t>(n);
            void * p = nullptr;
            pool_malloc(&p, nb, stream);
            ptr = static_cast<T *>(p);
        }
        count = n;
    }
    void release()
    {
        if (ptr != nullptr)
        {
            if (stream != nullptr)
            {
                (void)hipFreeAsync(ptr, stream);
            }
            else
            {
                (void)hipFree(ptr);
            }
            ptr = nullptr;
        }
        count = 0;
        stream = nullptr;
    }
    size_t bytes() const { return sizeof(T) * static_cast<size_t>(count); }
};

// The library's live streams: with the last one the pools are emptied.
inline std::atomic<int64_t> & live_streams()
{
    static std::atomic<int64_t> n{0};
    return n;
}

// A non-blocking stream at the default priority, synchronised and destroyed
// last: a handle declares it before its buffers, so they are freed on it
// while it still exists.
struct StreamHolder
{
    hipStream_t s = nullptr;
    StreamHolder()
    {
        SC_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        ++live_streams();
    }
    ~StreamHolder()
    {
        (void)hipStreamSynchronize(s);
        (void)hipStreamDestroy(s);
        if (--live_streams() == 0)
        {
            for (int dev = 0; dev < POOL_DEVICES; ++dev)
            {
                if (hipMemPool_t const pool = pool_slot(dev).load(std::memory_order_acquire))
                {
                    (void)hipMemPoolTrimTo(pool, 0);
                }
            }
        }
    }
    StreamHolder(StreamHolder const &) = delete;
    StreamHolder & operator=(StreamHolder const &) = delete;
};

// Between a pageable host array and device memory, ordered after the work on
// the stream and complete on return (transfer.hip).
void copy_down(void * host, void const * device, size_t nb, hipStream_t s);
void copy_up(void * device, void const * host, size_t nb, hipStream_t s);

inline unsigned grid_for(int64_t n, unsigned block)
{
    int64_t const g = (n + block - 1) / block;
    return static_cast<unsigned>(g < 1 ? 1 : g);
}

// gfx950 dispatches consecutive workgroups round-robin over its 8 XCDs, each
// with its own L2.  Remap the hardware block id so that every XCD works on
// one contiguous range of blocks: neighbour gathers of adjacent cells then
// hit the same L2.
__device__ inline unsigned xcd_block(unsigned b, unsigned nblk)
{
    constexpr unsigned NXCD = 8;
    unsigned const full = (nblk / NXCD) * NXCD;
    if (b >= full)
    {
        return b;
    }
    unsigned const per = nblk / NXCD;
    return (b % NXCD) * per + b / NXCD;
}

} /* end namespace scamd */
