// The planner's choices on the CPU: a Context with an MI355X's limits and no
// device (test infrastructure, called by tests/test_planner.py).
#include <memory>

#include "runtime.hpp"

using namespace mtgp;

namespace {
Context *make() {
    auto *c = new Context();
    c->cus = 256;
    // Workgroups per CU of each layout by the occupancy calculator.
    static const int limit[2][4][4] = {{{32, 32, 16, 8}, {24, 24, 16, 8}, {16, 16, 13, 4}, {0, 0, 0, 0}},
                                       {{16, 16, 15, 7}, {13, 13, 8, 7}, {7, 7, 5, 3}, {30, 30, 30, 30}}};
    for (int b = 0; b < 2; b++)
        for (int cls = 0; cls < 4; cls++)
            for (int lay = 0; lay < 4; lay++)
                c->blocks_per_cu[b][cls][lay] = limit[b][cls][lay];
    return c;
}
std::vector<GridGroup> group(int bits, int cls, int mexp, int n, const uint64_t *numbers) {
    GridGroup g;
    g.bits = bits;
    g.cls = cls;
    g.mexp = mexp;
    g.layouts = bits == 64 && cls == 3 ? 3 : 15;
    g.numbers.assign(numbers, numbers + n);
    return {g};
}
uint64_t sum(int n, const uint64_t *numbers) {
    uint64_t s = 0;
    for (int k = 0; k < n; k++)
        s += numbers[k];
    return s;
}
}  // namespace

extern "C" {

int planner_sizes(int bits, int cls, int mexp, int n, const uint64_t *numbers, uint64_t *out, int cap) {
    std::unique_ptr<Context> c(make());
    const auto v = one_round_sizes(*c, sum(n, numbers), group(bits, cls, mexp, n, numbers), 12 * c->cus);
    for (int k = 0; k < cap && k < (int)v.size(); k++)
        out[k] = v[(size_t)k];
    return (int)v.size();
}

double planner_ns(int bits, int cls, int mexp, int n, const uint64_t *numbers, uint64_t cell) {
    std::unique_ptr<Context> c(make());
    int64_t cells;
    return one_round_ns(*c, group(bits, cls, mexp, n, numbers), cell, cells);
}

// Workgroups per CU of a later launch of `cells` cells in the class's default
// layout (to *layout), after the autotuner chose (tuned_layout, tuned).
int planner_tuned(int bits, int cls, int tuned_layout, int tuned, int one_round, int cells, int *layout) {
    std::unique_ptr<Context> c(make());
    c->keep_tuned(bits, cls, tuned_layout, tuned, one_round != 0, true);
    const int mask = bits == 64 && cls == 3 ? 3 : 15;
    *layout = one_round ? c->layout_one_round_for(bits, cls, mask, cells, 1 << 16, (uint64_t)cells << 16)
                        : c->layout_for(bits, cls, mask);
    return c->launch_per_cu(bits, cls, *layout, cells, one_round != 0);
}

// The layout of a launch of equal cells, of one the model made (1) or a jump
// cache's grid (2) or any other (0); *fits as launch_layout has it.
int planner_layout(int bits, int cls, int mask, int cells, uint64_t cell, int grid, int *fits) {
    std::unique_ptr<Context> c(make());
    bool f;
    const int lay = c->launch_layout(bits, cls, mask, cells, cell, (uint64_t)cells * cell, grid == 1, grid == 2, f);
    *fits = f;
    return lay;
}

// Offsets and sizes of a jump's workspace.
void planner_jump_space(const uint64_t *bytes, uint64_t *out) {
    const JumpSpace W(bytes[0], bytes[1], bytes[2], bytes[3]);
    const uint64_t v[] = {W.o_coef, W.o_in, W.o_out, W.o_parts, W.device_bytes, W.host_bytes};
    for (int k = 0; k < 6; k++)
        out[k] = v[k];
}

// The one-round grid's cell size.
uint64_t planner_cell(int bits, int cls, int mexp, int n, const uint64_t *numbers) {
    std::unique_ptr<Context> c(make());
    uint64_t S1 = 0, S2 = 0;
    double frac = 0;
    auto_grid(*c, sum(n, numbers), n, group(bits, cls, mexp, n, numbers), 12 * c->cus, 1e300, 1, S1, S2, frac);
    return S1;
}
}
