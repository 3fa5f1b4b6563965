"""generate() calls that repeat their requests: work lists are kept for both
state slots, so the stream has to continue over many calls, over a state set
from outside between them, with generators that fall out of step, and over
other requests in between.  Whole numbers: every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [700, 90001])
def test_repeated_requests_continue_the_streams(mtgp, oracle, count):
    print("generate: repeated requests of %d numbers" % count, flush=True)
    specs = [(32, 11213, 4), (64, 23209, 6), (32, 44497, 1)]
    gs = mtgp.GenSet(specs)
    gs.init_seed([1, 2, 3])
    ps = [oracle.params(*s) for s in specs]
    ws = [oracle.init_state(p, 1 + g) for g, p in enumerate(ps)]
    bufs = [mtgp.DeviceBuffer(count * s[0] // 8) for s in specs]
    both, one = [(0, 0, count, 0, bufs[0]), (1, 0, count, 3, bufs[1]), (2, 0, count, 0, bufs[2])], [(1, 0, 5, 0, bufs[1])]

    def step(reqs):
        gs.generate(reqs)
        for g, _, n, skip, buf in reqs:
            if skip:
                _, ws[g] = oracle.generate(ps[g], ws[g], 0, skip)
            want, ws[g] = oracle.generate(ps[g], ws[g], 0, n)
            assert (buf.to_host(want.dtype, n) == want).all(), g
            assert (gs.state(g) == ws[g]).all(), g

    for _ in range(4):
        step(both)
    step(one)  # generator 1 is now one slot ahead of the others
    for _ in range(3):
        step(both)
    ws[2] = oracle.init_state(ps[2], 77)
    gs.set_state(2, ws[2])
    for _ in range(3):
        step(both)
    gs.jump(0, mtgp.jump_hex(32, 11213, 4, 1000))  # flips generator 0's slot outside of generate
    _, ws[0] = oracle.generate(ps[0], ws[0], 0, 1000)
    for _ in range(5):
        step(both)
