"""A server's batches of few cells (one to a few per class, at the cells'
edges) run in the step-time model's layouts; their numbers against the
oracle.  Whole numbers: every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELL = 1 << 17


@pytest.mark.parametrize("bits,mexp", [(32, 11213), (32, 23209), (64, 23209), (64, 44497)])
def test_batches_at_the_edges_of_cells(mtgp, oracle, bits, mexp):
    print("serve: MTGP%d-%d around the cell size" % (bits, mexp), flush=True)
    gs = mtgp.GenSet([(bits, mexp, 2), (bits, mexp, 5)])
    gs.init_seed([21, 22])
    ps = [oracle.params(bits, mexp, i) for i in (2, 5)]
    ws = [oracle.init_state(p, 21 + g) for g, p in enumerate(ps)]
    srv = mtgp.Server(gs, arena_bytes=64 << 20)
    for sizes in [(CELL,), (CELL - 1, 2, CELL + 1), (3 * CELL + 5, 1, 255)]:
        sent = {}
        for k, n in enumerate(sizes):
            g = k % 2
            sent[srv.submit(g, "uint", n, k)] = (g, n, k)
        got = {}
        while len(got) < len(sent):
            for c in srv.poll(wait_ms=100):
                got[c["ticket"]] = c
        for t in sorted(sent):
            g, n, skip = sent[t]
            if skip:
                _, ws[g] = oracle.generate(ps[g], ws[g], 0, skip)
            want, ws[g] = oracle.generate(ps[g], ws[g], 0, n)
            host = np.empty(n, want.dtype)
            mtgp.memcpy_dtoh(host, got[t]["out"])
            assert (host == want).all(), (g, n)
            srv.release(t)
