"""Automatic grids of dynamic-creator sets in every layout they admit: numbers,
and the windows that a commit leaves, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gens,count", [(32, 5, 200003), (64, 40, 9001), (64, 3, 500009)])
def test_numbers_and_committed_windows(mtgp, oracle, bits, gens, count):
    print("one-round grid: %d x MTGP%d-DC, %d numbers" % (gens, bits, count), flush=True)
    from pyoracle import Oracle
    from test_dc import _record
    recs = [mtgp.dc_params(bits, i % 200) for i in range(gens)]
    gs = mtgp.GenSet(recs)
    gs.init_seed([9 + g for g in range(gens)])
    dt, eb = (np.uint32, 4) if bits == 32 else (np.uint64, 8)
    buf = mtgp.DeviceBuffer(count * gens * eb)
    lens = [count - 37 * (g % 5) for g in range(gens)]
    plan = gs.plan([(g, 0, n, 0, buf.address(count * g * eb)) for g, n in enumerate(lens)])
    some = sorted({0, 1, gens // 2, gens - 1})
    ps = {g: Oracle.params_from_record(bits, _record(recs[g])) for g in some}
    want = {g: oracle.generate(p, oracle.init_state(p, 9 + g), 0, lens[g]) for g, p in ps.items()}
    for layout in (None, 1, 2, 3):
        if layout is not None:
            plan.configure(layout=layout)
        ran = {L["layout"] for L in plan.launches()}
        assert ran == ({1} if bits == 64 else {layout} if layout is not None else ran)
        buf.from_host(np.full(count * gens * eb, 0x5A, np.uint8))
        plan.launch()
        mtgp.synchronize()
        got = buf.to_host(dt, count * gens).reshape(gens, count)
        for g in some:
            assert (got[g, :lens[g]] == want[g][0]).all(), (layout, g)
    plan.commit()
    for g in some:
        assert (gs.state(g) == want[g][1]).all(), g
