"""One-round grids on the GPU against the oracle: the layout and the number of
cells follow the step-time model from a single short stream (no jumps) to many
long ones, and every layout of a plan writes the same numbers.  Whole numbers:
every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DC = "dc"


@pytest.mark.parametrize("bits,mexp,gens,count", [(32, 11213, 1, 4097), (32, 11213, 1, 1000003), (32, 11213, 137, 20011),
                                                  (32, 11213, 300, 70001), (32, 23209, 3, 300007), (32, 44497, 2, 500009),
                                                  (64, 23209, 1, 800011), (64, 23209, 600, 5003), (64, 44497, 9, 60013),
                                                  (32, DC, 5, 200003), (64, DC, 40, 9001)])
def test_model_grid(mtgp, oracle, bits, mexp, gens, count):
    print("one-round grid: %d x MTGP%d-%s, %d numbers" % (gens, bits, mexp, count), flush=True)
    specs = [mtgp.dc_params(bits, i % 200) if mexp == DC else (bits, mexp, i % 128) for i in range(gens)]
    gs = mtgp.GenSet(specs)
    gs.init_seed([9 + g for g in range(gens)])
    eb = bits // 8
    buf = mtgp.DeviceBuffer((count + 1) * gens * eb)
    lens = [count - 37 * (g % 5) for g in range(gens)]
    reqs = [(g, 0, n, 0, buf.address((count + 1) * g * eb)) for g, n in enumerate(lens)]
    plan = gs.plan(reqs)
    first, layouts = None, {L["layout"] for L in plan.launches()}
    for layout in [None, 1, 2, 3]:
        if layout is not None:
            plan.configure(layout=layout)
        buf.from_host(np.full((count + 1) * gens * eb, 0x5A, np.uint8))
        plan.launch()
        mtgp.synchronize()
        got = buf.to_host(np.uint32 if bits == 32 else np.uint64, (count + 1) * gens).reshape(gens, count + 1)
        if first is None:
            first = got.copy()
        assert (got == first).all(), layout
    plan.commit()
    guard = int.from_bytes(b"\x5a" * eb, "little")
    for g in sorted({0, gens // 2, gens - 1}):
        r = specs[g]
        p = oracle.params(*r) if mexp != DC else None
        assert (first[g, lens[g]:] == guard).all()
        if p is None:
            one = mtgp.GenSet([r])
            one.init_seed([9 + g])
            out = mtgp.DeviceBuffer(lens[g] * eb)
            one.plan([(0, 0, lens[g], 0, out)], segment=1 << 20).launch()
            mtgp.synchronize()
            assert (out.to_host(first.dtype, lens[g]) == first[g, :lens[g]]).all()
            assert (gs.state(g) != 0).any() and layouts
            continue
        want, w = oracle.generate(p, oracle.init_state(p, 9 + g), 0, lens[g])
        assert (first[g, :lens[g]] == want).all(), g
        assert (gs.state(g) == w).all(), g
