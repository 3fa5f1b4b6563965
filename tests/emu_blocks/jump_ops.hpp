// Stand-in for mtgp_amd/csrc/jump_ops.hpp: the same values in plain C++.
#pragma once
#include <stdint.h>

namespace mtgp {

inline uint32_t funnel32(uint32_t hi, uint32_t lo, uint32_t s) {
    return (uint32_t)((((uint64_t)hi << 32) | lo) >> (s & 31));
}

inline uint32_t wave_uniform(uint32_t v) { return v; }
inline uint32_t opaque(uint32_t v) { return v; }

template <int CT>
inline void interleave_step() {}
template <int P>
inline void wave_priority() {}

template <int D>
inline uint32_t lane_xor(uint32_t v) {
    return emu_lane_value<uint32_t>(v, (threadIdx.x & 63u) ^ (uint32_t)D);
}

inline void swap_halves(uint32_t &a, uint32_t &b) {
    const uint32_t l = threadIdx.x & 63u;
    const uint32_t b_low = emu_lane_value<uint32_t>(b, l & 31);
    const uint32_t a_high = emu_lane_value<uint32_t>(a, l | 32);
    if (l >= 32)
        a = b_low;
    else
        b = a_high;
}

// fp4 (e2m1) codes of 0 and 1.0 only: the operands hold nothing else.
inline float emu_fp4(uint32_t code) { return code == 2 ? 1.0f : code == 0 ? 0.0f : 1e30f; }

// The 32 x 32 x 64 product of one wave, with the operand and result layout
// of the matrix-core instruction.
inline mfma_v16f mfma_bits_32x32x64(mfma_v8i a, mfma_v8i b, mfma_v16f acc) {
    static uint32_t A[16][64][4], B[16][64][4];
    const int w = (int)threadIdx.x / 64, L = (int)threadIdx.x % 64;
    for (int v = 0; v < 4; v++) {
        A[w][L][v] = (uint32_t)a[v];
        B[w][L][v] = (uint32_t)b[v];
    }
    emu_wave_sync();
    mfma_v16f r = acc;
    for (int i = 0; i < 16; i++) {
        const int m = 8 * (i / 4) + 4 * (L / 32) + i % 4, n = L % 32;
        float s = 0.0f;
        for (int g = 0; g < 2; g++)
            for (int t = 0; t < 32; t++)
                s += emu_fp4(A[w][m + 32 * g][t / 8] >> (4 * (t % 8)) & 15) *
                     emu_fp4(B[w][n + 32 * g][t / 8] >> (4 * (t % 8)) & 15);
        r[i] += s;
    }
    emu_wave_sync();
    return r;
}

}  // namespace mtgp
