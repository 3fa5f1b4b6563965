"""Launches of about one to a few rounds of one cell per generator, at the
edges of the rule that gives them layout 1 in one round or layout 3 in
several, against layout 1 and the oracle.  Whole numbers: every comparison is
exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,mexp,gens,count", [(32, 11213, 2049, 33), (32, 11213, 4096, 1030), (32, 11213, 4097, 1030),
                                                  (32, 11213, 2600, 40001), (32, 23209, 3073, 2049), (32, 44497, 1030, 1025),
                                                  (64, 23209, 1800, 515), (64, 44497, 1793, 700)])
def test_many_cells(mtgp, oracle, bits, mexp, gens, count):
    print("many cells: %d x MTGP%d-%d, %d numbers" % (gens, bits, mexp, count), flush=True)
    gs = mtgp.GenSet([(bits, mexp, i % 128) for i in range(gens)])
    gs.init_seed([5 + g for g in range(gens)])
    dt, eb = (np.uint32, 4) if bits == 32 else (np.uint64, 8)
    buf = mtgp.DeviceBuffer((count + 1) * gens * eb)
    lens = [count - g % 7 for g in range(gens)]
    plan = gs.plan([(g, 0, n, 0, buf.address((count + 1) * g * eb)) for g, n in enumerate(lens)], segment=1 << 30)
    got = []
    for layout in (None, 1):
        if layout is not None:
            plan.configure(layout=layout)
        for _ in range(2):  # (the work queue is left as it was found)
            buf.from_host(np.full((count + 1) * gens * eb, 0x5A, np.uint8))
            plan.launch()
        mtgp.synchronize()
        got.append(buf.to_host(dt, (count + 1) * gens).reshape(gens, count + 1))
    assert (got[0] == got[1]).all()
    plan.commit()
    for g in (0, 1, gens // 2, gens - 2, gens - 1):
        p = oracle.params(bits, mexp, g % 128)
        want, w = oracle.generate(p, oracle.init_state(p, 5 + g), 0, lens[g])
        assert (got[0][g, :lens[g]] == want).all(), g
        assert (got[0][g, lens[g]:] == int.from_bytes(b"\x5a" * eb, "little")).all(), g
        assert (gs.state(g) == w).all(), g
