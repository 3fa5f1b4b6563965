"""The planner's choices on the CPU, against an MI355X's occupancy limits
(tests/planner): which cell sizes a one-round grid is chosen from, that
streams of nearby lengths are cut alike, so that their jump polynomials are in
the tables that an earlier call left, and that an autotuned launch shape is
the one that later plans run.  Whole numbers throughout."""
import ctypes as C
import math
import os
import random
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "planner")
U64 = C.c_uint64
# Workgroups per CU that fit, by layout (as tests/planner/driver.cpp has them)
LIMITS = {(32, 0): (32, 32, 16, 8), (32, 1): (24, 24, 16, 8), (32, 2): (16, 16, 13, 4), (64, 0): (16, 16, 15, 7),
          (64, 1): (13, 13, 8, 7), (64, 2): (7, 7, 5, 3), (64, 3): (30, 30, 30, 30)}
# (word size, state class): MEXP
CLASSES = {(32, 0): 11213, (32, 1): 23209, (32, 2): 44497, (64, 0): 23209, (64, 1): 44497, (64, 2): 110503, (64, 3): 3217}


@pytest.fixture(scope="module")
def lib():
    subprocess.check_call(["make", "-s", "-C", HERE])
    lib = C.CDLL(os.path.join(HERE, "libplanner.so"))
    one = [C.c_int] * 4 + [C.POINTER(U64)]
    lib.planner_sizes.argtypes = one + [C.POINTER(U64), C.c_int]
    lib.planner_ns.argtypes, lib.planner_ns.restype = one + [U64], C.c_double
    lib.planner_cell.argtypes, lib.planner_cell.restype = one, U64
    lib.planner_layout.argtypes = [C.c_int] * 4 + [U64, C.c_int, C.POINTER(C.c_int)]
    return lib


def _args(key, numbers):
    return (*key, CLASSES[key], len(numbers), (U64 * len(numbers))(*numbers))


def _sizes(lib, key, numbers):
    out = (U64 * 256)()
    n = lib.planner_sizes(*_args(key, numbers), out, 256)
    assert 0 < n <= 256
    return list(out[:n])


def _is_table_size(v, steps=4):
    while v >= 2 * steps:
        if v % 2:
            return False
        v //= 2
    return v >= steps


def _cell(lib, key, numbers):
    return lib.planner_cell(*_args(key, numbers))


@pytest.mark.parametrize("key", CLASSES)
def test_each_size_is_priced_once(lib, key):
    for numbers in ([1], [1000], [4096], [4097], [10**6], [1 << 24], [20000] * 200, [1000] * 128, [10**7, 5], [300007] * 3):
        sizes = _sizes(lib, key, numbers)
        assert len(set(sizes)) == len(sizes) and sizes == sorted(sizes, reverse=True), numbers
        # one cell per generator is among them, once
        assert sizes[0] >= max(numbers) and all(s < max(numbers) for s in sizes[1:]), numbers
        assert all(s >= 4096 and s % 256 == 0 for s in sizes)
        best = min(lib.planner_ns(*_args(key, numbers), s) for s in sizes
                   if s == sizes[0] or sum(-(-n // s) for n in numbers) <= 12 * 256)
        assert lib.planner_ns(*_args(key, numbers), _cell(lib, key, numbers)) == best


@pytest.mark.parametrize("key", CLASSES)
@pytest.mark.parametrize("n", [10**6, 1 << 24])
def test_nearby_lengths_share_a_grid(lib, key, n):
    """40 lengths of one stream within 2%: two cell sizes at most."""
    rng = random.Random(n)
    cells = {_cell(lib, key, [n - rng.randrange(n // 50)]) for _ in range(40)}
    assert len(cells) <= 2, cells


@pytest.mark.parametrize("key", CLASSES)
def test_streams_of_many_cells_take_table_sizes(lib, key):
    rng = random.Random(3)
    for lo, hi in ((10**5, 10**6), (10**6, 10**7), (10**7, 10**8)):
        cells = set()
        for _ in range(60):
            n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
            S = _cell(lib, key, [n])
            assert n // S < 3 or _is_table_size(S), (n, S)  # (2 cells stay 2 or more)
            if n // S >= 3:
                cells.add(S)
        assert len(cells) <= 14, cells  # 4 an octave over a decade


@pytest.mark.parametrize("gens,parts", [(2, 4), (16, 4), (17, 16), (64, 16)])
def test_sets_take_table_sizes_for_many_short_cells(lib, gens, parts):
    """From `parts` cells each on, of 2^17 numbers at most; the rounding may
    cost one cell in 17."""
    n = 1 << 22 if gens < 17 else 1 << 20
    sizes = _sizes(lib, (64, 0), [n + 1] * gens)
    assert all(_is_table_size(s, 16) for s in sizes if n // s >= parts + parts // 4 and s <= 7 << 14)
    assert any(not _is_table_size(s, 16) for s in sizes if 1 < n // s < parts), sizes
    sizes = _sizes(lib, (64, 0), [1 << 25] * 64)
    assert any(s > 1 << 17 and not _is_table_size(s, 16) for s in sizes)


@pytest.mark.parametrize("key", CLASSES)
@pytest.mark.parametrize("gens,n", [(2, 500000), (3, 2 * 10**6), (8, 400000)])
def test_nearby_lengths_of_few_streams_share_a_grid(lib, key, gens, n):
    rng = random.Random(n)
    cells = {_cell(lib, key, [n - rng.randrange(n // 50)] * gens) for _ in range(40)}
    cells = {S for S in cells if n // S >= 5 and S <= 7 << 14}
    assert len(cells) <= 3, cells


@pytest.mark.parametrize("key", CLASSES)
def test_later_launches_run_what_the_autotuner_measured(lib, key):
    """Every (layout, workgroups per CU) that the tuner tries, over launches of
    several rounds: at, below and beyond two rounds of it."""
    for layout in (1,) if key == (64, 3) else (0, 1, 2, 3):
        for per_cu in (2, 4, 6, 8, 12, 16):
            got = C.c_int()
            for cells in (256 * per_cu + 1, 300 * per_cu, 512 * per_cu, 512 * per_cu + 1, 5000 * per_cu):
                n = lib.planner_tuned(*key, layout, per_cu, 0, cells, C.byref(got))
                assert got.value == layout
                assert n == min(per_cu, LIMITS[key][layout]), (layout, per_cu, cells)


@pytest.mark.parametrize("lists,coef,window,parts", [(256, 128, 1404, 1408), (256, 1408, 1404, 15488),
                                                     (512, 4000 * 128, 13816, 4000 * 13824), (256, 1, 1, 128 << 20)])
def test_the_host_stages_no_partial_windows(lib, lists, coef, window, parts):
    out = (U64 * 6)()
    lib.planner_jump_space((U64 * 4)(lists, coef, window, parts), out)
    o_coef, o_in, o_out, o_parts, device, host = out
    assert all(o % 256 == 0 for o in (o_coef, o_in, o_out, o_parts))
    assert lists <= o_coef and o_coef + coef <= o_in and o_in + window <= o_out and o_out + window <= o_parts
    assert device == o_parts + parts and host <= lists + coef + 2 * window + 4 * 256


def _layout(lib, key, cells, cell, grid=0, mask=None):
    fits = C.c_int()
    mask = (3 if key == (64, 3) else 15) if mask is None else mask
    return lib.planner_layout(*key, mask, cells, cell, grid, C.byref(fits)), fits.value


@pytest.mark.parametrize("key", CLASSES)
def test_launches_of_several_rounds(lib, key):
    """Long cells take the widest layout that the sets admit; cells that layout
    1 holds in one round (12 per CU, 8 in the narrow class, and up to half as
    many again) and that are short stay in layout 1."""
    top = 1 if key == (64, 3) else 3
    one = 256 * min(8 if key == (64, 3) else 12, LIMITS[key][1])
    edge = min(3 * one // 2, 256 * LIMITS[key][1])
    assert _layout(lib, key, 100 * one, 1 << 17) == (top, 0)
    assert _layout(lib, key, edge, 4096) == (1, 0)
    assert _layout(lib, key, edge + 1, 4096) == (top, 0)
    assert _layout(lib, key, edge, 1 << 22) == (top, 0)
    for mask, lay in ((3, 1), (7, min(top, 2))):
        assert _layout(lib, key, 100 * one, 1 << 17, mask=mask & (3 if top == 1 else 15))[0] == lay


def test_short_cells_in_one_round_of_layout_1(lib):
    """The measured line: 4096 MTGP32-11213 cells of 2^12, 2^14, 2^17."""
    assert [_layout(lib, (32, 0), 4096, 1 << k)[0] for k in (12, 14, 17)] == [1, 1, 3]


@pytest.mark.parametrize("key", CLASSES)
def test_grids_of_one_round(lib, key):
    """A jump cache's grid runs as the model's while it is one round of it."""
    for cells in (1, 64, 256, 512):
        model = _layout(lib, key, cells, 1 << 17, 1)
        assert model[1] == 1 and _layout(lib, key, cells, 1 << 17, 2) == model
        if key != (64, 3):
            assert model[0] == 3 or cells > 256  # few cells: the shortest chain
    assert _layout(lib, key, 256 * 16 * 12, 1 << 17, 2)[1] == 0
    assert _layout(lib, key, 256 * 16 * 12, 1 << 17, 1)[1] == 1
