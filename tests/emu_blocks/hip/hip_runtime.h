// CPU stand-in for <hip/hip_runtime.h> for the blocked jump kernels: a
// workgroup runs as blockDim.x host threads, __syncthreads() is a real
// barrier over them, and cross-lane operations use a barrier of their own
// wave, so waves may run different trip counts between workgroup barriers.
// Workgroups of a launch run one after another; shared memory is a
// function-local static.  Test infrastructure only.
#pragma once
#include <stdint.h>
#include <string.h>

#include <barrier>
#include <memory>
#include <thread>
#include <vector>

#include "hip_runtime_api.h"

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __noinline__ __attribute__((noinline))
#define __shared__ static
#define __launch_bounds__(...)

struct emu_idx {
    uint32_t x = 0, y = 0, z = 0;
};
inline thread_local emu_idx threadIdx, blockIdx;
inline emu_idx gridDim, blockDim;

struct emu_block {
    std::barrier<> *bar = nullptr;
    std::barrier<> *wave[16] = {};
    uint64_t slots[1024];
};
inline emu_block g_emu_block;

inline void __syncthreads() { g_emu_block.bar->arrive_and_wait(); }
inline void emu_wave_sync() { g_emu_block.wave[threadIdx.x / 64]->arrive_and_wait(); }

// v of lane `src` of the caller's wave.
template <class T>
inline T emu_lane_value(T v, uint32_t src) {
    g_emu_block.slots[threadIdx.x] = (uint64_t)v;
    emu_wave_sync();
    T r = (T)g_emu_block.slots[(threadIdx.x & ~63u) + src];
    emu_wave_sync();
    return r;
}

inline uint32_t __float_as_uint(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    return u;
}

template <class... P, class... A>
inline void emu_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t, hipStream_t, A... args) {
    gridDim.x = grid.x;
    blockDim.x = block.x;
    for (uint32_t b = 0; b < grid.x; b++) {
        std::barrier<> bar((ptrdiff_t)block.x);
        g_emu_block.bar = &bar;
        std::vector<std::unique_ptr<std::barrier<>>> waves;
        for (uint32_t w = 0; w < block.x / 64; w++) {
            waves.push_back(std::make_unique<std::barrier<>>(64));
            g_emu_block.wave[w] = waves.back().get();
        }
        std::vector<std::thread> lanes;
        for (uint32_t t = 0; t < block.x; t++)
            lanes.emplace_back([=] {
                threadIdx.x = t;
                blockIdx.x = b;
                kernel(args...);
            });
        for (auto &th : lanes)
            th.join();
    }
}
#define hipLaunchKernelGGL emu_launch
