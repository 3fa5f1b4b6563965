"""The blocked matrix-core jump kernels (jump_blocks.hip) run on the CPU:
partial windows and folds against plain word XORs of the oracle's sequence,
for every state class at the edges of tiles and word groups.  Whole numbers:
every comparison is exact."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import pyemu

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu_blocks")
BLOCK, COLS, GROUP = 1024, 64, 16
GROUPS = np.dtype([("state_in", "<u8"), ("coef", "<u8"), ("parts", "<u8"), ("out", "<u8"), ("out_stride", "<u8"),
                   ("ncols", "<i4"), ("ch", "<i4"), ("param", "<i4"), ("n", "<i4"), ("pad", "<u8")])
TILE = np.dtype([("group", "<i4"), ("c0", "<i4"), ("param", "<i4"), ("plane", "<i4")])
SHARE = np.dtype([("tile0", "<i4"), ("tile1", "<i4"), ("g0", "<i4"), ("g1", "<i4"), ("first", TILE)])
FOLD = np.dtype([("group", "<i4"), ("b", "<i4")])
SETS = [(32, 11213, 3, 0), (32, 23209, 7, 1), (32, 44497, 1, 2), (64, 23209, 2, 0), (64, 44497, 5, 1), (64, 110503, 9, 2),
        (64, "dc", 172, 3)]


@pytest.fixture(scope="module")
def emu():
    subprocess.check_call(["make", "-s", "-C", HERE])
    lib = C.CDLL(os.path.join(HERE, "libblocks_emu.so"), mode=os.RTLD_LOCAL)
    vp = C.c_void_p
    lib.emu_jump_tiles.argtypes = [C.c_int, C.c_int, vp, vp, vp, C.c_int, vp]
    lib.emu_jump_folds.argtypes = [C.c_int, C.c_int, C.c_int, vp, vp, C.c_int, vp]
    return lib


def _set(mtgp, bits, mexp, idx):
    """Parameter record and device record of a table or dynamic-creator set."""
    r = mtgp.dc_params(bits, idx) if mexp == "dc" else mtgp.params(bits, mexp, idx)
    flt = r.flt_tmp_tbl if bits == 32 else r.dbl_tmp_tbl
    rec = [r.mexp, r.pos, r.sh1, r.sh2, *r.tbl, *r.tmp_tbl, *flt, r.mask]
    return r, pyemu.devparam(bits, rec)


def _sequence(bits, r, w, count):
    """w continued by `count` words of its recursion."""
    n, pos, W = len(w), r.pos, w.dtype.type
    s = np.concatenate([w, np.zeros(count, w.dtype)])
    tbl = np.array(list(r.tbl), w.dtype)
    for k in range(0, count, n - pos):
        m = min(n - pos, count - k)
        x = (s[k:k + m] & W(r.mask)) ^ s[k + 1:k + 1 + m]
        y = s[k + pos:k + pos + m]
        if bits == 32:
            v = x ^ (x << W(r.sh1)) ^ (y >> W(r.sh2))
        else:
            xh, xl = (x >> W(32)).astype(np.uint32), x.astype(np.uint32)
            s1, s2 = np.uint32(r.sh1), np.uint32(r.sh2)
            vh = xl ^ (xl << s1) ^ ((y >> W(32)).astype(np.uint32) >> s2)
            vl = xh ^ (xh << s1) ^ (y.astype(np.uint32) >> s2)
            v = (vh.astype(W) << W(32)) | vl.astype(W)
        s[n + k:n + k + m] = v ^ tbl[(v & W(15)).astype(np.int64)]
    return s


def _planes(bits, a):
    """Words (.., n) as 32-bit planes, each padded to whole word groups."""
    n = a.shape[-1]
    pad = [(0, 0)] * (a.ndim - 1) + [(0, -n % GROUP)]
    if bits == 32:
        return np.pad(a, pad)
    return np.concatenate([np.pad((a >> np.uint64(32)).astype(np.uint32), pad), np.pad(a.astype(np.uint32), pad)], -1)


@pytest.mark.parametrize("bits,mexp,idx,cls", SETS)
def test_tiles(emu, mtgp, bits, mexp, idx, cls):
    """Partial windows of a full and a partial column tile for the first, a
    middle and the last word groups, in shares of one tile and across tiles
    and planes; columns hold single coefficients (first,
    last, word edges), everything, nothing and random bits."""
    r, dev = _set(mtgp, bits, mexp, idx)
    rng = np.random.default_rng(idx + bits)
    n = r.mexp // bits + 1
    w = rng.integers(0, 2**bits, n, dtype=np.uint32 if bits == 32 else np.uint64)
    ncols = 70 + idx % 2 * 30
    bit = np.zeros((ncols, BLOCK), bool)
    for c, k in enumerate((0, 1, 31, 32, 63, 64, 1022, 1023)):
        bit[c, k] = True
    bit[8] = True
    bit[10:] = rng.random((ncols - 10, BLOCK)) < 0.5
    coef = np.packbits(bit, axis=1, bitorder="little").view(np.uint32).copy()
    pw = (n + GROUP - 1) // GROUP * GROUP
    parts = np.full((ncols, bits // 32 * pw), 0xA5A5A5A5, np.uint32)
    g = np.zeros(1, GROUPS)
    g["state_in"], g["coef"], g["parts"] = w.ctypes.data, coef.ctypes.data, parts.ctypes.data
    g["ncols"], g["ch"], g["n"] = ncols, 5, n
    last = pw // GROUP
    # tiles by plane and column; shares within one tile, from the last groups
    # of one tile to the first of the next, and (MTGP64) across the planes
    tiles = np.array([(0, c0, 0, q) for q in range(bits // 32) for c0 in (0, COLS)], TILE)
    runs = [(0, 0, 0, 1), (0, 1, last - 1, 1), (1, 1, 3, 4), (1, 1, last - 2, last)]
    if bits == 64:
        runs += [(1, 2, last - 1, 1), (2, 3, last - 1, 2)]
    shares = np.array([(*q, tiles[q[0]]) for q in runs], SHARE)
    assert emu.emu_jump_tiles(bits, cls, g.ctypes.data, tiles.ctypes.data, shares.ctypes.data, len(shares),
                              dev.ctypes.data) == 0
    s = _sequence(bits, r, w, BLOCK)
    want = np.zeros((ncols, n), w.dtype)
    for c in range(ncols):
        for k in np.nonzero(bit[c])[0]:
            want[c] ^= s[k:k + n]
    want = _planes(bits, want)
    seen = np.zeros(parts.shape, bool)
    for t0, t1, first, end in runs:
        for t in range(t0, t1 + 1):
            c0, plane = int(tiles[t]["c0"]), int(tiles[t]["plane"])
            cols = slice(c0, min(c0 + COLS, ncols))
            for j in range(GROUP * (first if t == t0 else 0), GROUP * (end if t == t1 else last)):
                at = plane * pw + j
                seen[cols, at] = True
                if j < n:
                    assert (parts[cols, at] == want[cols, at]).all(), (t, j)
    assert (parts[~seen] == 0xA5A5A5A5).all(), "written outside the tiles"


@pytest.mark.parametrize("bits,mexp,idx,cls", SETS)
@pytest.mark.parametrize("ch", [1, 2, 4])
def test_folds(emu, mtgp, bits, mexp, idx, cls, ch):
    """Horner's rule over 1, 2 and 4 partial windows, for every step the class
    has kernels of."""
    r, dev = _set(mtgp, bits, mexp, idx)
    rng = np.random.default_rng(idx + ch)
    n = r.mexp // bits + 1
    nj = 2
    P = rng.integers(0, 2**bits, (nj, ch, n), dtype=np.uint32 if bits == 32 else np.uint64)
    parts = _planes(bits, P).copy()
    want = []
    for b in range(nj):
        v = P[b, ch - 1]
        for a in range(ch - 2, -1, -1):
            v = _sequence(bits, r, v, BLOCK)[BLOCK:] ^ P[b, a]
        want.append(v)
    step = emu.emu_jump_step(bits, cls, n, r.pos)
    assert step <= n - r.pos and BLOCK % step == 0
    while step >= (128 if cls == 3 else 256):
        out = np.zeros((nj, n + 3), P.dtype)
        g = np.zeros(1, GROUPS)
        g["parts"], g["out"], g["out_stride"] = parts.ctypes.data, out.ctypes.data, out.strides[0]
        g["ncols"], g["ch"], g["n"] = nj * ch, ch, n
        folds = np.array([(0, 0), (0, 1)], FOLD)
        assert emu.emu_jump_folds(bits, cls, step, g.ctypes.data, folds.ctypes.data, nj, dev.ctypes.data) == 0
        assert (out[:, :n] == np.array(want)).all() and (out[:, n:] == 0).all(), step
        step //= 2
