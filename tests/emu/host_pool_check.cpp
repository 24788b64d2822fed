// The server's host blocks (host_pool.hpp): what a request of a size holds,
// what it is given back, and how much the pool keeps.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <new>
#include <vector>

#include "host_pool.hpp"
using namespace pano;

// operator new fails while g_fail_from counts down to 0 and after
static std::atomic<int> g_fail_from{1 << 30};
void* operator new(size_t n) {
    if (g_fail_from.fetch_sub(1) <= 0) throw std::bad_alloc();
    void* p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static int fails = 0;
#define CHECK(cond, ...)                 \
    do {                                 \
        if (!(cond)) {                   \
            ++fails;                     \
            printf("FAIL %s: ", #cond);  \
            printf(__VA_ARGS__);         \
            printf("\n");                \
        }                                \
    } while (0)

int main() {
    // a queued request holds its velocity and little more
    for (size_t n : {size_t(16), size_t(4096), size_t(33280), size_t(263168), size_t(1 << 20), (size_t(4) << 20) - 4,
                     size_t(4) << 20, size_t(8396800), size_t(203) << 20}) {
        HostPool P;
        HostBlock b(&P, n);
        CHECK(b.p && b.cap >= n, "%zu bytes", n);
        CHECK(b.cap <= n + n / 2 + 4096, "%zu bytes hold %zu", n, b.cap);
        memset(b.p, 1, n);
    }
    // a block that is given back serves requests of about its size only
    {
        HostPool P;
        const size_t n = 12 << 20;
        void* first;
        {
            HostBlock b(&P, n);
            first = b.p;
        }
        HostBlock small(&P, 33280), half(&P, n / 2 - (2 << 20)), same(&P, n - 1000);
        CHECK(small.p != first && half.p != first, "a smaller request took the block");
        CHECK(same.p == first, "the next request of the size did not");
    }
    {
        HostPool P;
        void* first;
        {
            HostBlock b(&P, 100);
            first = b.p;
        }
        HostBlock same(&P, 60);
        CHECK(same.p == first, "a small block is not used again");
    }
    // moved blocks are given back once
    {
        HostPool P;
        std::vector<HostBlock> v;
        for (int i = 0; i < 40; ++i) {
            HostBlock b(&P, size_t(1000) * (i + 1));
            memset(b.p, i, size_t(1000) * (i + 1));
            HostBlock c;
            c = std::move(b);
            v.push_back(std::move(c));
        }
        v.clear();
    }
    // copies around the chunk limits
    for (size_t n : {size_t(0), size_t(1), kParCopyMin - 1, kParCopyMin, kParCopyMin + 1, kParCopyMin + 12345}) {
        std::vector<unsigned char> a(n), b(n + 1, 7);
        for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 131 + (i >> 9));
        par_copy((char*)b.data(), (const char*)a.data(), n);
        CHECK(memcmp(a.data(), b.data(), n) == 0 && b[n] == 7, "copy of %zu bytes", n);
    }
    // no host memory for a thread's start: the copy is whole all the same
    for (int k = 0; k < 3; ++k) {
        const size_t n = kParCopyMin + 777;
        std::vector<char> a(n, 3), b(n, 0);
        g_fail_from = k;
        par_copy(b.data(), a.data(), n);
        g_fail_from = 1 << 30;
        CHECK(a == b, "copy with %d allocations left", k);
    }
    // none for the pool's own record: the block is freed, not kept
    {
        HostPool P;
        {
            HostBlock b(&P, 5000);
            g_fail_from = 0;
        }
        g_fail_from = 1 << 30;
        HostBlock c(&P, 5000);
        CHECK(c.p != nullptr, "no block");
    }
    printf("%d failures\n", fails);
    return fails != 0;
}
