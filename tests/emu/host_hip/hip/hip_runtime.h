// Host stand-ins for what the solver's headers and cg_cluster.hip use of HIP,
// so that the kernel's own source is built by a host compiler and its threads
// are run by the scheduler of cluster_emu.cpp. A workgroup is an OS thread
// (its __shared__ variables are thread_local), a GPU thread one of its fibers.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) alignas(n)
#define __shared__ thread_local

struct dim3 {
    unsigned x, y, z;
    constexpr dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
constexpr hipError_t hipSuccess = 0;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return "emulated"; }

// ---- the emulated GPU thread (cluster_emu.cpp) -------------------------------------
extern thread_local dim3 threadIdx, blockIdx, blockDim, gridDim;

void __syncthreads();
bool __any(bool);
int emu_dpp(int old, int v, int ctrl, int row_mask, int bank_mask, bool bound);
int emu_readlane(int v, int lane);
void emu_waitcnt();                                              // this wave's stores have completed
void emu_store(void* p, const void* v, size_t n);                // in flight until then, or for some time
void emu_load(const void* p, void* v, size_t n);
bool emu_launch(dim3 grid, dim3 block, size_t lds, void (*body)(void*), void* arg);

#define __HIP_MEMORY_SCOPE_AGENT 0
template <typename V>
inline V emu_atomic_load(const V* p) {
    V v;
    emu_load(p, &v, sizeof(V));
    return v;
}
template <typename V>
inline void emu_atomic_store(V* p, V v) {
    emu_store(p, &v, sizeof(V));
}
#define __hip_atomic_load(p, order, scope) emu_atomic_load(p)
#define __hip_atomic_store(p, v, order, scope) emu_atomic_store(p, v)
#define __builtin_amdgcn_update_dpp emu_dpp
#define __builtin_amdgcn_readlane emu_readlane
inline int __popc(unsigned v) { return __builtin_popcount(v); }

inline long long __double_as_longlong(double v) {
    long long b;
    memcpy(&b, &v, 8);
    return b;
}
inline double __longlong_as_double(long long b) {
    double v;
    memcpy(&v, &b, 8);
    return v;
}

// lane swaps that other kernels of the headers use; none of them is run here
struct EmuPair {
    int v[2];
    int operator[](int i) const { return v[i]; }
};
inline EmuPair __builtin_amdgcn_permlane32_swap(int, int, bool, bool) { abort(); }
inline EmuPair __builtin_amdgcn_permlane16_swap(int, int, bool, bool) { abort(); }

// the only inline assembly is the wait for the wave's stores
#define asm emu_waitcnt(); if (0) __asm__

template <typename K, typename... A>
inline void emu_kernel_launch(K kernel, dim3 grid, dim3 block, size_t lds, A... args) {
    auto call = [=] { kernel(args...); };
    emu_launch(grid, block, lds, [](void* c) { (*static_cast<decltype(call)*>(c))(); }, &call);
}
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    emu_kernel_launch(kernel, grid, block, lds, __VA_ARGS__)
template <typename... A>
inline void hipExtLaunchKernelGGL(A...) { abort(); }
