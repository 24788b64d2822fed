// Host memory of the server: blocks for queued velocities and copies of large
// ranges.
#pragma once

#include <sys/mman.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <thread>

namespace pano {

// memcpy of large host ranges by a few threads. One thread copies into memory
// it touches for the first time at 10 to 14 GB/s (page faults), four at three
// times that. Threads that cannot be started leave their part to the caller.
constexpr size_t kParCopyMin = size_t(4) << 20;
inline void par_copy(char* dst, const char* src, size_t n) {
    constexpr int N = 4;
    if (n < kParCopyMin) {
        memcpy(dst, src, n);
        return;
    }
    const size_t part = ((n / N + 4095) / 4096) * 4096;
    std::thread th[N - 1];
    for (int i = 1; i < N; ++i) {
        const size_t a = std::min(n, i * part), b = i == N - 1 ? n : std::min(n, (i + 1) * part);
        try {
            th[i - 1] = std::thread([=] { memcpy(dst + a, src + a, b - a); });
        } catch (...) {  // no thread, or no memory for one
            memcpy(dst + a, src + a, b - a);
        }
    }
    memcpy(dst, src, std::min(n, part));
    for (std::thread& t : th)
        if (t.joinable()) t.join();
}

// Host blocks for the velocities of queued requests. A block that a request
// gives back is kept for the next one, up to kKeep bytes: a new allocation of
// this size is page faults on its first write (the copy at submit took 190 ms
// for 0.9 GB into new vectors). Blocks from kParCopyMin on are whole huge pages,
// smaller ones whole pages: ten thousand queued 64 x 64 requests hold 360 MB
// (a huge page each would be 20 GB).
class HostPool {
public:
    ~HostPool() {
        for (auto& b : free_) ::free(b.second);
    }
    // a block of at least n bytes (nullptr: no memory); *cap its size
    void* take(size_t n, size_t* cap) {
        const size_t page = n < kParCopyMin ? kPage : kHuge, want = (n + page - 1) / page * page;
        auto it = free_.lower_bound(n);
        if (it != free_.end() && it->first <= 2 * want) {
            void* p = it->second;
            *cap = it->first;
            kept_ -= it->first;
            free_.erase(it);
            return p;
        }
        *cap = want;
        void* p = nullptr;
        if (posix_memalign(&p, page, want) != 0) return nullptr;
        if (page == kHuge) (void)madvise(p, want, MADV_HUGEPAGE);
        return p;
    }
    void give(void* p, size_t cap) {
        if (kept_ + cap > kKeep) {
            ::free(p);
            return;
        }
        try {
            free_.emplace(cap, p);
        } catch (...) {  // no memory to remember it by (destructors call this)
            ::free(p);
            return;
        }
        kept_ += cap;
    }

private:
    static constexpr size_t kPage = 4096, kHuge = size_t(2) << 20, kKeep = size_t(1) << 30;
    std::multimap<size_t, void*> free_;
    size_t kept_ = 0;
};

// A block of the pool, given back when it goes.
struct HostBlock {
    HostPool* pool = nullptr;
    void* p = nullptr;
    size_t cap = 0;
    HostBlock() = default;
    HostBlock(HostPool* pl, size_t n) : pool(pl) { p = pl->take(n, &cap); }
    HostBlock(HostBlock&& o) noexcept : pool(o.pool), p(o.p), cap(o.cap) { o.p = nullptr; }
    HostBlock& operator=(HostBlock&& o) noexcept {
        std::swap(pool, o.pool);
        std::swap(p, o.p);
        std::swap(cap, o.cap);
        return *this;
    }
    ~HostBlock() {
        if (p) pool->give(p, cap);
    }
};

}  // namespace pano
