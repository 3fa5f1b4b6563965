"""The word-XOR jump kernels (jump_mfma_min = 0) of every state class, MTGP64
and the dynamic-creator sets among them, against the oracle: plans launched
twice, a launch with more work items than workgroups (its work queue is left
as it was found), substreams by levels, and single jumps of host and device
windows, which are split over waves and combined.  Whole numbers: every
comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TABLE = [(32, 11213, 7), (32, 23209, 90), (32, 44497, 3), (64, 23209, 11), (64, 44497, 2), (64, 110503, 1)]
DC = [(32, "dc", 16), (64, "dc", 172)]


def _set(mtgp, oracle, spec):
    """What GenSet takes for `spec`, and the oracle's parameters."""
    bits, mexp, idx = spec
    if mexp != "dc":
        return spec, oracle.params(*spec)
    from test_dc import _record
    rec = mtgp.dc_params(bits, idx)
    return rec, type(oracle).params_from_record(bits, _record(rec))


@pytest.mark.parametrize("spec", TABLE + DC)
@pytest.mark.parametrize("cells", [2, 5, 6, 23])
def test_plans(mtgp, oracle, spec, cells):
    """cells - 1 jumps: one batch of up to four, a batch and one, several."""
    print("word-XOR jumps: MTGP%d-%s, %d cells" % (spec[0], spec[1], cells), flush=True)
    s, p = _set(mtgp, oracle, spec)
    gs = mtgp.GenSet([s] * 2)
    gs.init_seed([50, 51])
    count = 4096 * (cells - 1) + 777
    bufs = [mtgp.DeviceBuffer(count * spec[0] // 8) for _ in range(2)]
    with mtgp.tuning(jump_mfma_min=0):
        plan = gs.plan([(g, 0, count, 0, b) for g, b in enumerate(bufs)], segment=4096)
    assert plan.stats()["jumps"] == 2 * (cells - 1) and plan.stats()["matrix_jumps"] == 0
    # one jump launch and one of generation; blocked jumps have two
    assert plan.stats()["launches"] == 2
    assert gs.plan([(g, 0, count, 0, b) for g, b in enumerate(bufs)], segment=4096).stats()["launches"] == 3
    want = [oracle.generate(p, oracle.init_state(p, 50 + g), 0, count) for g in range(2)]
    for _ in range(2):
        for b, (e, _w) in zip(bufs, want):
            b.from_host(np.full(e.nbytes, 0x5A, np.uint8))
        plan.launch()
        mtgp.synchronize()
        for b, (e, _w) in zip(bufs, want):
            assert (b.to_host(e.dtype, count) == e).all()
    plan.commit()
    for g, (_e, w) in enumerate(want):
        assert (gs.state(g) == w).all()


@pytest.mark.parametrize("bits,mexp,gens", [(32, 11213, 8300), (64, 23209, 8300)])
def test_more_items_than_workgroups(mtgp, oracle, bits, mexp, gens):
    """One jump per generator: 8300 items for at most 32 workgroups on each of
    256 CUs, launched twice."""
    print("word-XOR jumps: %d items of MTGP%d-%d" % (gens, bits, mexp), flush=True)
    gs = mtgp.GenSet([(bits, mexp, g % 128) for g in range(gens)])
    gs.init_seed([7 + g for g in range(gens)], device=True)
    count, eb, dt = 4096 + 33, bits // 8, np.uint32 if bits == 32 else np.uint64
    room = 4352
    buf = mtgp.DeviceBuffer(gens * room * eb)
    with mtgp.tuning(jump_mfma_min=0):
        plan = gs.plan([(g, 0, count, 0, buf.address(g * room * eb)) for g in range(gens)], segment=4096)
    assert plan.stats()["jumps"] == gens
    some = (0, 1, gens // 2, 8191, 8192, gens - 1)
    want = {}
    for g in some:
        p = oracle.params(bits, mexp, g % 128)
        want[g] = oracle.generate(p, oracle.init_state(p, 7 + g), 0, count)
    got = []
    for _ in range(2):
        buf.from_host(np.full(gens * room * eb, 0x5A, np.uint8))
        plan.launch()
        mtgp.synchronize()
        got.append(buf.to_host(dt, gens * room).reshape(gens, room))
        for g in some:
            assert (got[-1][g, :count] == want[g][0]).all(), g
    assert (got[0] == got[1]).all()
    plan.commit()
    for g in some:
        assert (gs.state(g) == want[g][1]).all(), g


@pytest.mark.parametrize("spec,count", [((32, 23209, 5), 7), ((64, 23209, 5), 19), ((64, 110503, 5), 3),
                                        ((64, "dc", 199), 17)])
def test_substreams(mtgp, oracle, spec, count):
    print("word-XOR jumps: %d substreams of MTGP%d-%s" % (count, spec[0], spec[1]), flush=True)
    s, p = _set(mtgp, oracle, spec)
    js = mtgp.jump_hex(spec[0], record=s, steps=10**7) if spec[1] == "dc" else mtgp.jump_hex(*spec, 10**7)
    gs = mtgp.GenSet([s] * count)
    with mtgp.tuning(jump_mfma_min=0):
        for seed in (3, 4):
            w = oracle.init_state(p, seed)
            gs.substreams(w, js)
            for t in range(count):
                # (word 0's bits outside the mask are no state)
                got, mask = gs.state(t), w.dtype.type(p.mask)
                assert (got[1:] == w[1:]).all() and got[0] & mask == w[0] & mask, t
                w = oracle.jump(p, w, js)


@pytest.mark.parametrize("spec", TABLE + DC)
def test_single_jumps(mtgp, oracle, spec):
    """Polynomials of one to many chunks, applied to a host generator and to a
    device set: the zero polynomial, 1, x, a chunk's edges, and one of higher
    degree than the set's."""
    print("word-XOR jumps: single jumps of MTGP%d-%s" % (spec[0], spec[1]), flush=True)
    s, p = _set(mtgp, oracle, spec)
    rec = s if spec[1] == "dc" else None
    mexp = s.mexp if spec[1] == "dc" else spec[1]
    rng = np.random.default_rng(mexp)

    def hexs(coeffs):
        v = np.zeros(max(list(coeffs) + [0]) // 4 + 1, int)
        for k in coeffs:
            v[k // 4] |= 1 << (k % 4)
        return "".join("%x" % q for q in v)

    dense = [k for k in range(mexp) if rng.random() < 0.5]
    polys = [[], [0], [1], [1023], [1024], [2047, 2048], dense, dense[:1000] + [mexp + 3000]]
    G = mtgp.Generator32 if spec[0] == 32 else mtgp.Generator64
    with mtgp.tuning(jump_mfma_min=0):
        for k, cs in enumerate(polys):
            js = hexs(cs)
            g = G(record=rec, seed=5 + k) if rec is not None else G(mexp, spec[2], seed=5 + k)
            gs = mtgp.GenSet([s])
            gs.init_seed([5 + k])
            w = oracle.init_state(p, 5 + k)
            assert (g.window() == w).all()
            want = oracle.jump(p, w, js)
            g.fast_jump(js)
            assert (g.window() == want).all(), k
            gs.jump(0, js)
            assert (gs.state(0) == want).all(), k
