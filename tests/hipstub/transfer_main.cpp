/* Copies on a stream whose device is not the current one (test_transfer_host.py). */
#include "common.hpp"

#include <cstdio>
#include <vector>

namespace scamd
{
void set_last_error(int, std::string const &) {}
}

int main()
{
    using namespace scamd;
    size_t const n = 40u << 20;
    std::vector<char> a(n), b(n);
    for (size_t k = 0; k < n; ++k)
    {
        a[k] = static_cast<char>(k * 2654435761u >> 13);
    }
    int bad = 0;
    // Every lane of device 0 is made first, then device 1 copies.
    for (int dev = 0; dev < 2; ++dev)
    {
        (void)hipSetDevice(dev);
        StreamHolder sh;
        for (int current = 0; current < 2; ++current)
        {
            (void)hipSetDevice(current);
            for (int down = 0; down < 2; ++down)
            {
                std::vector<char> c(n);
                int const before = stub_copies();
                try
                {
                    down != 0 ? copy_down(c.data(), a.data(), n, sh.s) : copy_up(c.data(), a.data(), n, sh.s);
                }
                catch (std::exception const & e)
                {
                    std::printf("stream of %d, current %d, down %d: %s\n", dev, current, down, e.what());
                    ++bad;
                    continue;
                }
                int d = -1;
                (void)hipGetDevice(&d);
                bool const ok = c == a && d == current && stub_copies() - before > 1;
                std::printf("stream of %d, current %d, down %d: %s\n", dev, current, down, ok ? "ok" : "WRONG");
                bad += ok ? 0 : 1;
            }
        }
        (void)hipSetDevice(1 - dev);
        OnDevice const on(sh.s);
        StreamHolder other;
        bad += other.s->dev == dev ? 0 : 1;
    }
    return bad;
}
