"""Generation in cells of one word per lane and four waves (layout 3 of the
smallest classes), the library's kernels run on the CPU: around the step, the
window relocation after eight steps, unaligned outputs, partial start windows
and a segment chain.  Whole numbers: every comparison is exact."""
import numpy as np
import pytest

import pyemu
from test_kernel_emulation import _bits, _run


@pytest.fixture(scope="module")
def emu():
    return pyemu.load()


@pytest.mark.parametrize("bits,mexp,idx", [(32, 11213, 3), (32, 11213, 127), (64, 23209, 0), (64, 23209, 90)])
def test_one_word_cells(emu, oracle, bits, mexp, idx):
    p = oracle.params(bits, mexp, idx)
    assert p.n - p.pos >= 256
    eb, wd = bits // 8, np.uint32 if bits == 32 else np.uint64
    w0 = oracle.init_state(p, 7 + idx)
    counts = [(0, 1), (1, 255), (2, 256), (3, 257), (4, 2047), (0, 2049), (1, 0), (2, 4099)]
    items, keep = [], []
    for k, (kind, n) in enumerate(counts):
        raw = np.zeros((n + 16) * eb + 128, np.uint8)
        at = -raw.ctypes.data % 128 + eb * (5 * k % 16)
        sout = np.zeros_like(w0)
        items.append(dict(out=raw.ctypes.data + at, count=n, state_in=w0.ctypes.data, state_out=sout.ctypes.data,
                          param=pyemu.set_id(bits, mexp, idx), kind=kind, n=p.n))
        keep.append((raw, at, sout))
    parts = np.random.default_rng(idx).integers(0, np.iinfo(wd).max, (3, p.n), dtype=wd)
    parts[2] = w0 ^ parts[0] ^ parts[1]
    chain = [(0, 5), (None, 700), (2, 2300), (None, 3), (1, 257)]
    segs, outs, w = np.zeros(len(chain), pyemu.SEGMENT), [], w0
    for k, (kind, n) in enumerate(chain):
        raw = np.zeros((n + 16) * eb + 128, np.uint8)
        at = -raw.ctypes.data % 128 + eb * (3 * k % 16)
        segs[k] = (0 if kind is None else raw.ctypes.data + at, n, kind or 0, 0, 0)
        e, w = oracle.generate(p, w, kind or 0, n)
        outs.append((raw, at, e[:0] if kind is None else e))
    cout = np.zeros_like(w0)
    items.append(dict(state_in=parts.ctypes.data, state_out=cout.ctypes.data, param=pyemu.set_id(bits, mexp, idx),
                      segs=segs.ctypes.data, nsegs=len(chain), parts=3, part_bytes=p.n * eb, n=p.n))
    _run(emu, bits, items, 3, grid=4)
    for (kind, n), (raw, at, sout) in zip(counts, keep):
        e, we = oracle.generate(p, w0, kind, n)
        outs.append((raw, at, e))
        assert (sout == we).all(), (kind, n)
    for raw, at, e in outs:
        assert (_bits(raw[at:at + len(e) * eb].view(e.dtype)) == _bits(e)).all()
        assert not raw[:at].any() and not raw[at + len(e) * eb:].any(), "write outside the outputs"
    assert (cout == w).all()
