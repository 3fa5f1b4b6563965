"""The planner's choices on the CPU, against an MI355X's occupancy limits
(tests/planner): which cell sizes a one-round grid is chosen from."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "planner")
U64 = C.c_uint64
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
    return lib


def _args(key, numbers):
    return (*key, CLASSES[key], len(numbers), (U64 * len(numbers))(*numbers))


def _sizes(lib, key, numbers):
    out = (U64 * 256)()
    n = lib.planner_sizes(*_args(key, numbers), out, 256)
    assert 0 < n <= 256
    return list(out[:n])


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
