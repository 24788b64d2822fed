// The server's host blocks (host_pool.hpp): what a request of a size holds,
// what it is given back, and how much the pool keeps.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "host_pool.hpp"
using namespace pano;

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
    printf("%d failures\n", fails);
    return fails != 0;
}
