"""Blocked matrix-core jumps on the GPU against the oracle: plans of every
state class with one to many jumps per generator, a plan whose partial
windows need several rounds of launches, and substreams by levels and as one
group.  Whole numbers: every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SETS = [(32, 11213, 7), (32, 23209, 90), (32, 44497, 3), (64, 23209, 11), (64, 44497, 2), (64, 110503, 1)]


@pytest.mark.parametrize("cells", [2, 3, 8, 40])
def test_plans_of_every_class(mtgp, oracle, cells):
    """One generator per class in one plan, cells of 4096 numbers (cells - 1
    jumps each, the last cell partial)."""
    print("blocked jumps: %d cells per generator" % cells, flush=True)
    gs = mtgp.GenSet(SETS)
    gs.init_seed([50 + g for g in range(len(SETS))])
    count = 4096 * (cells - 1) + 777
    bufs = [mtgp.DeviceBuffer(count * s[0] // 8) for s in SETS]
    plan = gs.plan([(g, 0, count, 0, b) for g, b in enumerate(bufs)], segment=4096)
    assert plan.stats()["jumps"] == len(SETS) * (cells - 1)
    plan.launch()
    mtgp.synchronize()
    plan.commit()
    for g, (s, b) in enumerate(zip(SETS, bufs)):
        p = oracle.params(*s)
        want, w = oracle.generate(p, oracle.init_state(p, 50 + g), 0, count)
        assert (b.to_host(want.dtype, count) == want).all(), s
        assert (gs.state(g) == w).all(), s


def test_several_rounds(mtgp, oracle):
    """199 MTGP64-110503 jumps (1.5 MB of partial windows each) run in three
    rounds of launches that reuse the partial windows' memory."""
    print("blocked jumps: several rounds", flush=True)
    p = oracle.params(64, 110503, 4)
    gs = mtgp.GenSet([(64, 110503, 4)])
    gs.init_seed([99])
    count = 4096 * 200
    buf = mtgp.DeviceBuffer(count * 8)
    plan = gs.plan([(0, 0, count, 0, buf)], segment=4096)
    assert plan.stats()["launches"] == 2 * 3 + 1
    plan.launch()
    mtgp.synchronize()
    want, _ = oracle.generate(p, oracle.init_state(p, 99), 0, count)
    assert (buf.to_host(want.dtype, count) == want).all()


@pytest.mark.parametrize("bits,mexp,count", [(32, 11213, 1), (32, 11213, 2), (32, 11213, 70), (32, 11213, 257),
                                             (32, 44497, 6), (64, 23209, 4), (64, 23209, 19)])
def test_substreams(mtgp, oracle, bits, mexp, count):
    """Substream t = the base jumped t times by 10^7 steps, by levels (up to
    256 substreams and MTGP64) and as one group, twice from two bases."""
    print("blocked jumps: %d substreams of MTGP%d-%d" % (count, bits, mexp), flush=True)
    p = oracle.params(bits, mexp, 5)
    js = mtgp.jump_hex(bits, mexp, 5, 10**7)
    gs = mtgp.GenSet([(bits, mexp, 5)] * count)
    for seed in (3, 4):
        base = oracle.init_state(p, seed)
        gs.substreams(base, js)
        w = base
        for t in range(count):
            if t < 20 or t > count - 3:
                # (word 0's bits outside the mask are no state: they depend on
                # how the jump is composed)
                got, mask = gs.state(t), w.dtype.type(p.mask)
                assert (got[1:] == w[1:]).all() and got[0] & mask == w[0] & mask, t
            w = oracle.jump(p, w, js)


@pytest.mark.parametrize("bits,mexp", [(32, 11213), (32, 44497), (64, 23209), (64, 110503)])
def test_single_jumps(mtgp, oracle, bits, mexp):
    """Polynomials at the edges of the blocks, applied to a host generator and
    to a device set: the zero polynomial, 1, x, the last coefficient of a
    block and the first of the next, one block and a word, dense ones, and one
    of higher degree than the set's."""
    print("blocked jumps: single jumps of MTGP%d-%d" % (bits, mexp), flush=True)
    p = oracle.params(bits, mexp, 6)
    rng = np.random.default_rng(mexp)

    def hexs(coeffs):
        # four coefficients per character, the lowest ones first
        v = np.zeros(max(list(coeffs) + [0]) // 4 + 1, int)
        for k in coeffs:
            v[k // 4] |= 1 << (k % 4)
        return "".join("%x" % q for q in v)

    dense = [k for k in range(mexp) if rng.random() < 0.5]
    polys = [[], [0], [1], [1023], [1024], [0, 1023, 1024, 1055], dense, dense[:1000] + [mexp + 3000]]
    G = mtgp.Generator32 if bits == 32 else mtgp.Generator64
    for k, cs in enumerate(polys):
        s = hexs(cs)
        g = G(mexp, 6, seed=5 + k)
        gs = mtgp.GenSet([(bits, mexp, 6)])
        gs.init_seed([5 + k])
        w = oracle.init_state(p, 5 + k)
        assert (g.window() == w).all()
        want = oracle.jump(p, w, s)
        g.fast_jump(s)
        assert (g.window() == want).all(), k
        gs.jump(0, s)
        assert (gs.state(0) == want).all(), k
