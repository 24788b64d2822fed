// The server's fetch stage (fetch_stage.hpp) where a part of it cannot be had:
// all of it or nothing, and another try at the next fetch. Built with the
// stand-ins of host_hip/.
#include <cstdio>

static int g_left = 0, g_held = 0;  // calls that succeed, things held
#include <hip/hip_runtime.h>
constexpr unsigned hipEventDisableTiming = 2;
static hipError_t get(void** out) {
    if (g_left-- <= 0) return 2;
    ++g_held;
    *out = malloc(1);
    return hipSuccess;
}
static hipError_t give(void* p) {
    --g_held;
    free(p);
    return hipSuccess;
}
static hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return get(e); }
static hipError_t hipEventDestroy(hipEvent_t e) { return give(e); }
static hipError_t hipHostMalloc(void** p, size_t) { return get(p); }
static hipError_t hipHostFree(void* p) { return give(p); }

#include "fetch_stage.hpp"
using namespace pano;

int main() {
    int fails = 0;
    for (int k = 0; k <= 3; ++k) {
        FetchStage f;
        g_left = k;
        const bool made = f.make();
        if (made != (k == 3) || made != (f.p && f.ev[0] && f.ev[1]) || g_held != (made ? 3 : 0)) {
            ++fails;
            printf("FAIL %d calls succeed: made %d, %d held\n", k, made, g_held);
        }
        g_left = 3;
        if (!f.make() || !f.p || !f.ev[0] || !f.ev[1] || g_held != 3) {
            ++fails;
            printf("FAIL the next try after %d calls\n", k);
        }
    }
    if (g_held) ++fails, printf("FAIL %d left\n", g_held);
    printf("%d failures\n", fails);
    return fails != 0;
}
