/* The library's device memory pool (test_transfer_host.py). */
#include "common.hpp"

#include <cstdio>

namespace scamd
{
void set_last_error(int, std::string const &) {}
}

int main()
{
    using namespace scamd;
    StubMemory & m = stub_memory();
    constexpr int64_t GB = int64_t(1) << 30;
    int bad = 0;
    auto expect = [&](bool ok, char const * what)
    {
        std::printf("%s: %s\n", what, ok ? "ok" : "WRONG");
        bad += ok ? 0 : 1;
    };
    m.def[0].keep = 123; // what the application has set
    {
        StreamHolder one, two;
        {
            AllocScope const scope(one.s);
            DevBuf<char> a;
            a.alloc(12 * GB);
        }
        expect(m.def[0].keep == 123, "the default pool's threshold is the application's");
        expect(m.def[0].reserved == 0, "the default pool is not used");
        expect(m.taken[0] == uint64_t(12 * GB), "freed memory is kept");
        // Neither kind of allocation finds 8 GB free beside the kept 12.
        {
            DevBuf<char> b; // no scope: hipMalloc
            b.alloc(8 * GB);
            expect(m.taken[0] == uint64_t(8 * GB), "hipMalloc gets the kept memory");
        }
        {
            AllocScope const scope(one.s);
            DevBuf<char> c;
            c.alloc(6 * GB);
        }
        {
            AllocScope const scope(two.s);
            DevBuf<char> d, e;
            d.alloc(5 * GB);
            e.alloc(11 * GB);
            expect(m.taken[0] == uint64_t(16 * GB), "the device is full");
            DevBuf<char> f;
            bool refused = false;
            try
            {
                f.alloc(1);
            }
            catch (std::exception const &)
            {
                refused = true;
            }
            expect(refused, "an allocation that cannot be had is refused");
        }
        // A stream of another device allocates there.
        (void)hipSetDevice(1);
        StreamHolder far;
        (void)hipSetDevice(0);
        AllocScope const scope(far.s);
        DevBuf<char> g;
        g.alloc(GB);
        expect(m.taken[1] == uint64_t(GB), "the stream's device counts");
    }
    expect(m.taken[0] == 0 && m.taken[1] == 0, "the last stream gives all back");
    return bad;
}
