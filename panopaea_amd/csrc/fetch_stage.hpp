// The two pinned halves through which the server's large fetches run, each
// with the event that its copy has ended.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace pano {

constexpr size_t kFetchChunk = size_t(8) << 20;

struct FetchStage {
    char* p = nullptr;  // 2 * kFetchChunk bytes
    hipEvent_t ev[2] = {nullptr, nullptr};
    FetchStage() = default;
    FetchStage(const FetchStage&) = delete;
    FetchStage& operator=(const FetchStage&) = delete;
    ~FetchStage() { drop(); }

    // whether there is a stage: made at the first call that gets all of it
    bool make() {
        if (p) return true;
        void* mem = nullptr;
        if (hipEventCreateWithFlags(&ev[0], hipEventDisableTiming) == hipSuccess &&
            hipEventCreateWithFlags(&ev[1], hipEventDisableTiming) == hipSuccess &&
            hipHostMalloc(&mem, 2 * kFetchChunk) == hipSuccess) {
            p = static_cast<char*>(mem);
            return true;
        }
        (void)hipGetLastError();
        drop();
        return false;
    }
    void drop() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        for (hipEvent_t& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
};

}  // namespace pano
