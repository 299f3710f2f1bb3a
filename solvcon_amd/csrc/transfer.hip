/*
 * Copies between device tables and pageable host arrays (the host mirrors).
 *
 * A plain hipMemcpyAsync on pageable memory goes through the runtime's own
 * staging on one thread: 17 GB/s to the host and 28 GB/s from it on 144 MB,
 * less where the host pages are new.  Large copies therefore go in chunks
 * through pinned buffers kept here: several threads each move one contiguous
 * share, the link filling one of a thread's two buffers while the thread
 * empties the other: 40 GB/s and 39 GB/s.
 */

#include "common.hpp"

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <memory>
#include <new>
#include <thread>
#include <vector>

namespace scamd
{
namespace
{

constexpr size_t CHUNK = 2u << 20;
constexpr int LANES = 8;      // pinned buffer pairs per device: 32 MB at most
constexpr int PER_COPY = 4;   // threads of one copy

struct Lane
{
    int dev = 0;
    char * buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};

    Lane() = default;
    Lane(Lane const &) = delete;
    Lane & operator=(Lane const &) = delete;
    ~Lane()
    {
        for (int b = 0; b < 2; ++b)
        {
            if (ev[b] != nullptr)
            {
                (void)hipEventDestroy(ev[b]);
            }
        }
        if (buf[0] != nullptr)
        {
            (void)hipHostFree(buf[0]);
        }
    }
    bool open(int device)
    {
        dev = device;
        void * p = nullptr;
        if (hipHostMalloc(&p, 2 * CHUNK, hipHostMallocDefault) != hipSuccess)
        {
            (void)hipGetLastError();
            return false;
        }
        buf[0] = static_cast<char *>(p);
        buf[1] = buf[0] + CHUNK;
        for (int b = 0; b < 2; ++b)
        {
            if (hipEventCreateWithFlags(&ev[b], hipEventDisableTiming) != hipSuccess)
            {
                (void)hipGetLastError();
                return false;
            }
        }
        return true;
    }
};

struct Lanes
{
    std::mutex mu;
    std::vector<Lane *> idle;
    std::map<int, int> made; // by device
    size_t total = 0;
};

// Never destroyed: the process's end takes it, after the HIP runtime.
Lanes & lanes()
{
    static Lanes * const l = new Lanes;
    return *l;
}

// The lanes of one copy, given back when it ends: at most n, fewer (or none)
// when others use them.
struct Taken
{
    std::vector<Lane *> v;
    Taken(int n, int dev)
    {
        Lanes & l = lanes();
        std::lock_guard<std::mutex> const lock(l.mu);
        // All that may throw comes first: no lane is lost, and giving them
        // back allocates nothing.
        int & made = l.made[dev];
        v.reserve(static_cast<size_t>(n));
        l.idle.reserve(l.total + static_cast<size_t>(n));
        for (size_t k = 0; k < l.idle.size() && static_cast<int>(v.size()) < n;)
        {
            if (l.idle[k]->dev == dev)
            {
                v.push_back(l.idle[k]);
                l.idle.erase(l.idle.begin() + static_cast<std::ptrdiff_t>(k));
            }
            else
            {
                ++k;
            }
        }
        while (static_cast<int>(v.size()) < n && made < LANES)
        {
            std::unique_ptr<Lane> lane(new (std::nothrow) Lane);
            if (lane == nullptr || !lane->open(dev))
            {
                break;
            }
            v.push_back(lane.release());
            ++made;
            ++l.total;
        }
    }
    ~Taken()
    {
        Lanes & l = lanes();
        std::lock_guard<std::mutex> const lock(l.mu);
        l.idle.insert(l.idle.end(), v.begin(), v.end());
    }
    Taken(Taken const &) = delete;
    Taken & operator=(Taken const &) = delete;
};

// One lane's share.  Returns the first error; nothing of the lane is in flight
// when it returns.
hipError_t share(Lane & l, bool down, char * host, char * device, size_t nb, hipStream_t s)
{
    hipError_t e = hipSuccess;
    bool used[2] = {false, false};
    auto wait = [&](int b)
    {
        if (used[b])
        {
            hipError_t const w = hipEventSynchronize(l.ev[b]);
            e = e == hipSuccess ? w : e;
            used[b] = false;
        }
    };
    size_t const n = (nb + CHUNK - 1) / CHUNK;
    auto size = [&](size_t k) { return std::min(CHUNK, nb - k * CHUNK); };
    for (size_t k = 0; k < n + 1 && e == hipSuccess; ++k)
    {
        int const b = static_cast<int>(k & 1);
        if (k < n)
        {
            char * const h = host + k * CHUNK;
            char * const d = device + k * CHUNK;
            if (!down)
            {
                wait(b);
                std::memcpy(l.buf[b], h, size(k));
            }
            hipError_t const c = down ? hipMemcpyAsync(l.buf[b], d, size(k), hipMemcpyDeviceToHost, s)
                                      : hipMemcpyAsync(d, l.buf[b], size(k), hipMemcpyHostToDevice, s);
            e = e == hipSuccess ? c : e;
            if (c == hipSuccess)
            {
                hipError_t const r = hipEventRecord(l.ev[b], s);
                e = e == hipSuccess ? r : e;
                used[b] = r == hipSuccess;
            }
        }
        if (down && k > 0)
        {
            wait(1 - b);
            if (e == hipSuccess)
            {
                std::memcpy(host + (k - 1) * CHUNK, l.buf[1 - b], size(k - 1));
            }
        }
    }
    wait(0);
    wait(1);
    if (e != hipSuccess)
    {
        (void)hipStreamSynchronize(s); // a copy without its event may still run
    }
    return e;
}

void copy_host(bool down, void * host, void * device, size_t nb, hipStream_t s)
{
    // Where the threads pay for themselves (12 MB down: 418 us against 674, up:
    // 381 against 331; 4.8 MB down: 271 against 285).
    size_t const least = down ? 4u << 20 : 32u << 20;
    int const want = nb < least ? 0 : static_cast<int>(std::min<size_t>(PER_COPY, 1 + nb / (2 * CHUNK)));
    OnDevice const on(s);
    int const dev = on.dev;
    Taken const lanes(want, dev);
    int const n = static_cast<int>(lanes.v.size());
    if (n == 0)
    {
        SC_HIP(down ? hipMemcpyAsync(host, device, nb, hipMemcpyDeviceToHost, s)
                    : hipMemcpyAsync(device, host, nb, hipMemcpyHostToDevice, s));
        SC_HIP(hipStreamSynchronize(s));
        return;
    }
    char * const h = static_cast<char *>(host);
    char * const d = static_cast<char *>(device);
    auto cut = [&](int k) { return k == n ? nb : nb / n * k / 4096 * 4096; };
    std::vector<hipError_t> err(static_cast<size_t>(n), hipSuccess);
    auto work = [&](int k, bool own)
    {
        hipError_t e = own ? hipSuccess : hipSetDevice(dev);
        if (e == hipSuccess)
        {
            e = share(*lanes.v[k], down, h + cut(k), d + cut(k), cut(k + 1) - cut(k), s);
        }
        err[k] = e;
    };
    std::vector<std::thread> th;
    int started = 1;
    try
    {
        th.reserve(static_cast<size_t>(n));
        for (; started < n; ++started)
        {
            th.emplace_back(work, started, false);
        }
    }
    catch (std::exception const &)
    {
        // No more threads: this one does the rest.
    }
    work(0, true);
    for (int k = started; k < n; ++k)
    {
        work(k, true);
    }
    for (auto & t : th)
    {
        t.join();
    }
    for (hipError_t e : err)
    {
        SC_HIP(e);
    }
    SC_HIP(hipStreamSynchronize(s));
}

} /* end namespace */

void copy_down(void * host, void const * device, size_t nb, hipStream_t s)
{
    copy_host(true, host, const_cast<void *>(device), nb, s);
}

void copy_up(void * device, void const * host, size_t nb, hipStream_t s)
{
    copy_host(false, const_cast<void *>(host), device, nb, s);
}

} /* end namespace scamd */
