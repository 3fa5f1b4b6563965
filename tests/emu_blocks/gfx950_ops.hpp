// Stand-in for mtgp_amd/csrc/gfx950_ops.hpp: what the blocked jump kernels
// use of it, in plain C++ (wave-wide operations per 64 threads).
#pragma once
#include <stdint.h>

namespace mtgp {

inline uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) { return a ^ b ^ c; }

typedef int mfma_v8i __attribute__((ext_vector_type(8)));
typedef float mfma_v16f __attribute__((ext_vector_type(16)));

}  // namespace mtgp
