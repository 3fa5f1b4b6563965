"""One-round grids whose cell sizes several lengths share: streams of 1 to a
few cells, and of many, each length followed by a shorter and a longer one that
find the first one's jump polynomials in the kept tables, against the oracle.
Whole numbers: every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,mexp,gens,lengths", [
    (32, 11213, 1, (12289, 12288, 13001, 250000, 255000, 244444, 1500000, 1530001)),
    (32, 44497, 1, (100003, 104000, 98765, 1200001, 1250000)),
    (64, 23209, 1, (65537, 70001, 64000, 900001)),
    (64, 110503, 1, (60001, 61440, 300007, 310000)),
    (32, 23209, 3, (400003, 420001, 390000)),
    (64, 44497, 5, (150001, 160000))])
def test_lengths_after_one_another(mtgp, oracle, bits, mexp, gens, lengths):
    print("table grids: %d x MTGP%d-%d" % (gens, bits, mexp), flush=True)
    specs = [(bits, mexp, 7 + g) for g in range(gens)]
    gs = mtgp.GenSet(specs)
    gs.init_seed([31 + g for g in range(gens)])
    ps = [oracle.params(*s) for s in specs]
    ws = [oracle.init_state(p, 31 + g) for g, p in enumerate(ps)]
    dt, eb = (np.uint32, 4) if bits == 32 else (np.uint64, 8)
    room = max(lengths) + 1
    buf = mtgp.DeviceBuffer(room * gens * eb)
    for n in lengths:
        buf.from_host(np.full(room * gens * eb, 0x5A, np.uint8))
        gs.generate([(g, 0, n - 3 * g, 0, buf.address(room * g * eb)) for g in range(gens)])
        got = buf.to_host(dt, room * gens).reshape(gens, room)
        for g in range(gens):
            want, ws[g] = oracle.generate(ps[g], ws[g], 0, n - 3 * g)
            assert (got[g, :n - 3 * g] == want).all(), (n, g)
            assert (got[g, n - 3 * g:] == int.from_bytes(b"\x5a" * eb, "little")).all(), (n, g)
            assert (gs.state(g) == ws[g]).all(), (n, g)
