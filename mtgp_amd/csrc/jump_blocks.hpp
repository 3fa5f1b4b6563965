// jump_blocks.hpp -- work lists and launch interface of jump_blocks.hip:
// jumps on the matrix cores in blocks of kJbBlock coefficients.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include "common.hpp"

namespace mtgp {

// Coefficients per block.  A jump polynomial c is cut into `ch` blocks of
// kJbBlock coefficients; block a of a jump gives the partial window
// P_a[j] = XOR_{i : c[kJbBlock a + i] = 1} w[i + j] over the base's own
// sequence w, and the jumped window is P_{ch-1} advanced by kJbBlock numbers,
// XORed with P_{ch-2}, advanced again, and so on down to P_0.
constexpr int kJbBlock = 1024;
constexpr int kJbWords = kJbBlock / 32;  // coefficient words per block
constexpr int kJbCols = 64;              // partial windows (columns) per tile, at most
constexpr int kJbGroup = 16;             // window words per word group (one pass of a workgroup)

// All jumps of one base window.  Column c = b * ch + a is block a of jump b.
struct alignas(16) JumpBlocks {
    uint64_t state_in;    // base window (N words)
    uint64_t coef;        // uint32_t[ncols][kJbWords]: column c's coefficients
    uint64_t parts;       // uint32_t[ncols][part_words]: partial windows, the 32-bit
                          // planes (one for MTGP32; high, low for MTGP64) jb_plane_words(n) apart
    uint64_t out;         // jump b's window at out + b * out_stride
    uint64_t out_stride;  // bytes
    int32_t ncols, ch, param, n;
    uint64_t pad;
};
static_assert(sizeof(JumpBlocks) == 64, "JumpBlocks layout");

// Words of one plane of a partial window (a whole number of word groups).
inline int jb_plane_words(int n) { return (n + kJbGroup - 1) / kJbGroup * kJbGroup; }
inline int jb_part_words(int bits, int n) { return bits / 32 * jb_plane_words(n); }
// Blocks of a polynomial of `coeffs` coefficients.
inline int jb_blocks(int64_t coeffs) { return (int)(coeffs <= kJbBlock ? 1 : (coeffs + kJbBlock - 1) / kJbBlock); }

// Columns [c0, c0 + kJbCols) of a group (as far as it has them), all word
// groups of plane `plane`.  A launch's tiles are ordered by group, plane, c0.
struct alignas(16) JumpTile {
    int32_t group, c0, param, plane;
};
static_assert(sizeof(JumpTile) == 16, "JumpTile layout");

// One workgroup of the products: tiles [tile0, tile1] (both included), the
// first (a copy of it: one load less before the work starts) from word group
// g0 on, the last up to word group g1.
struct alignas(16) JumpShare {
    int32_t tile0, tile1, g0, g1;
    JumpTile first;
};
static_assert(sizeof(JumpShare) == 32, "JumpShare layout");

// One workgroup of the fold: jump b of a group.
struct JumpFold {
    int32_t group, b;
};

// Every group's set is of word size `bits` and class <= cls (kernels.hpp).
// The products of n_shares workgroups, then the folds of n_folds jumps, which
// advance `step` numbers at once (at most any set's jb_step).
hipError_t launch_jump_tiles(int bits, int cls, const JumpBlocks *groups, const JumpTile *tiles,
                             const JumpShare *shares, int n_shares, const DevParam *params, hipStream_t s);
hipError_t launch_jump_folds(int bits, int cls, int step, const JumpBlocks *groups, const JumpFold *folds, int n_folds,
                             const DevParam *params, hipStream_t s);
// Numbers the fold advances at once for a set: the largest of its class's
// steps that N - pos admits.
int jb_step(int bits, int cls, int n, int pos);

}  // namespace mtgp
