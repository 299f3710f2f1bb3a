/* Copies while host memory is short (test_transfer_host.py). */
#include "common.hpp"

#include <cstdio>
#include <new>
#include <vector>

namespace scamd
{
void set_last_error(int, std::string const &) {}
}

// The main thread's n-th allocation from now on fails (0: none does).
static thread_local int fail_at = 0;

static void * get(size_t n)
{
    if (fail_at > 0 && --fail_at == 0)
    {
        return nullptr;
    }
    return std::malloc(n);
}

void * operator new(size_t n)
{
    void * const p = get(n);
    return p != nullptr ? p : throw std::bad_alloc();
}
void * operator new(size_t n, std::nothrow_t const &) noexcept { return get(n); }
void operator delete(void * p) noexcept { std::free(p); }
void operator delete(void * p, size_t) noexcept { std::free(p); }

int main(int, char ** argv)
{
    using namespace scamd;
    size_t const n = 10u << 20;
    std::vector<char> a(n, 7), c(n);
    StreamHolder sh;
    fail_at = std::atoi(argv[1]);
    try
    {
        copy_down(c.data(), a.data(), n, sh.s);
    }
    catch (std::bad_alloc const &)
    {
    }
    fail_at = 0;
    // Afterwards the copy has its chunks and threads again.
    int bad = 0;
    c.assign(n, 0);
    int const before = stub_copies();
    copy_down(c.data(), a.data(), n, sh.s);
    bad += c == a && stub_copies() - before > 1 ? 0 : 1;
    std::printf("%d copies\n", stub_copies() - before);
    return bad;
}
