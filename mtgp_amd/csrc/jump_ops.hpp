// jump_ops.hpp -- single gfx950 instructions of the blocked jump kernels.
#pragma once
#include <stdint.h>

namespace mtgp {

// Low word of (hi:lo) >> s, s < 32 (v_alignbit_b32).
__device__ __forceinline__ uint32_t funnel32(uint32_t hi, uint32_t lo, uint32_t s) {
    return __builtin_amdgcn_alignbit(hi, lo, s);
}

// v, the same in every lane of the wave, as a scalar.
__device__ __forceinline__ uint32_t wave_uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// A scalar v, as a value the compiler knows nothing about.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+s"(v));
    return v;
}

// v of lane (lane ^ D), D = 1, 2, 4, 8 or 16, by register moves across lanes
// (no LDS access).
template <int D>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (D == 16) {
        // rows of 16 lanes: the odd rows of one copy with the even ones of the
        // other
        typedef uint32_t v2 __attribute__((ext_vector_type(2)));
        const v2 r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (threadIdx.x & 16) ? r[0] : r[1];
    } else if constexpr (D == 8) {
        return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);  // row_ror:8
    } else if constexpr (D == 4) {
        v = __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true);        // row_half_mirror: ^ 7
        return __builtin_amdgcn_mov_dpp(v, 0x1b, 0xf, 0xf, true);      // quad_perm 3,2,1,0: ^ 3
    } else if constexpr (D == 2) {
        return __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true);  // quad_perm 2,3,0,1
    } else {
        return __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
    }
}

// Scheduling of one product step with CT column tiles: its 4 CT matrix
// instructions in order, after each a few vector instructions of the next
// step's operands and an LDS read of the one after's; nothing moves across its
// end (the steps accumulate into the same registers, so two of them mixed
// would wait for each other's results).
template <int CT>
__device__ __forceinline__ void interleave_step() {
#pragma unroll
    for (int i = 0; i < 4 * CT; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);           // matrix
        __builtin_amdgcn_sched_group_barrier(0x002, 4 / CT + 1, 0);  // vector
        if (i < 2 + CT)
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Issue priority of this wave among those of its SIMD (0 .. 3).
template <int P>
__device__ __forceinline__ void wave_priority() {
    __builtin_amdgcn_s_setprio(P);
}

// Exchanges the upper 32 lanes of a with the lower 32 lanes of b.
__device__ __forceinline__ void swap_halves(uint32_t &a, uint32_t &b) {
    typedef uint32_t v2 __attribute__((ext_vector_type(2)));
    const v2 r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// acc + A B with A 32 x 64 and B 64 x 32 in fp4: lane L holds row L % 32 of A
// and column L % 32 of B, both for the 32 values of K group L / 32 (the same
// value index means the same k in both); acc[r] of lane L is row 8 (r / 4) +
// 4 (L / 32) + r % 4, column L % 32.  In the form without block scales: an
// 8-byte instruction with no scale registers.
__device__ __forceinline__ mfma_v16f mfma_bits_32x32x64(mfma_v8i a, mfma_v8i b, mfma_v16f acc) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 4, 4, 0, 0, 0, 0);
}

}  // namespace mtgp
