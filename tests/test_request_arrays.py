"""Request arrays for plans and generate calls: every field of every request, at
the edges of the blocks they are packed in, what ctypes converts by itself, what
it refuses, and no memory kept per distinct number of requests."""
import ctypes as C
import tracemalloc

import pytest


def _rows(arr, n):
    return [(r.gen, r.kind, r.count, r.skip, r.out or 0) for r in arr[:n]]


@pytest.mark.parametrize("n", [0, 1, 2, 127, 128, 129, 255, 256, 257, 1000])
def test_every_field(mtgp, n):
    want = [(k % 7, k % 5, 3 * k, 2**40 + k, 2**47 + 64 * k) for k in range(n)]
    assert _rows(mtgp._request_array(n, [v for row in want for v in row]), n) == want
    assert _rows(mtgp._requests(want), n) == want


def test_as_ctypes_converts_them(mtgp):
    # negative and wide numbers wrap, None is NULL, names are kinds
    reqs = [(k % 3, 0, k, 0, 4096 + k) for k in range(150)]
    reqs[140] = (-1, "close_open", -2, 2**64 + 5, None)
    got = _rows(mtgp._requests(reqs), 150)
    assert got[:140] == reqs[:140] and got[141:] == reqs[141:]
    assert got[140] == (-1, mtgp.KINDS["close_open"], 2**64 - 2, 5, 0)


@pytest.mark.parametrize("bad", [1.5, "x", [1]])
def test_refused(mtgp, bad):
    with pytest.raises(TypeError):
        mtgp._requests([(0, 0, 1, 0, 64)] * 129 + [(0, 0, bad, 0, 64)])


def test_no_memory_is_kept_per_number_of_requests(mtgp):
    fields = [0, 0, 1, 0, 4096] * 40100
    for m in range(1, 129):
        mtgp._request_array(m, fields[:5 * m])
    tracemalloc.start()
    try:
        for n in range(40000, 40100, 10):
            mtgp._request_array(n, fields[:5 * n])
        kept, _ = tracemalloc.get_traced_memory()
    finally:
        tracemalloc.stop()
    # (a format of 40000 requests alone is 5 * 40000 entries of 32 bytes)
    assert kept < 1 << 20, kept
