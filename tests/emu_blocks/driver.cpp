// Entry points of the blocked jump emulation library.
#include <vector>

#include "common.hpp"
#include "jump_blocks.hpp"
#include "kernels.hpp"

extern "C" int emu_jump_tiles(int bits, int cls, const mtgp::JumpBlocks *groups, const mtgp::JumpTile *tiles,
                              const mtgp::JumpShare *shares, int n, const mtgp::DevParam *params) {
    return mtgp::launch_jump_tiles(bits, cls, groups, tiles, shares, n, params, nullptr) == hipSuccess ? 0 : -1;
}

extern "C" int emu_jump_folds(int bits, int cls, int step, const mtgp::JumpBlocks *groups, const mtgp::JumpFold *folds,
                              int n, const mtgp::DevParam *params) {
    return mtgp::launch_jump_folds(bits, cls, step, groups, folds, n, params, nullptr) == hipSuccess ? 0 : -1;
}

extern "C" int emu_jump_step(int bits, int cls, int n, int pos) { return mtgp::jb_step(bits, cls, n, pos); }
