"""A plan of several rounds that the autotuner has run, made again: the same
launches (layout, grid) as were measured, and the oracle's numbers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,mexp,gens,count,segment", [(32, 11213, 64, 1 << 18, 4096), (64, 44497, 64, 1 << 17, 4096)])
def test_a_later_plan_runs_the_tuned_launches(mtgp, oracle, bits, mexp, gens, count, segment):
    print("autotune kept: %d x MTGP%d-%d" % (gens, bits, mexp), flush=True)
    gs = mtgp.GenSet([(bits, mexp, g) for g in range(gens)])
    gs.init_seed([3 + g for g in range(gens)])
    dt, eb = (np.uint32, 4) if bits == 32 else (np.uint64, 8)
    buf = mtgp.DeviceBuffer(gens * count * eb)
    reqs = [(g, 0, count, 0, buf.address(g * count * eb)) for g in range(gens)]
    first = gs.plan(reqs, segment=segment)
    first.autotune(reps=1)
    again = gs.plan(reqs, segment=segment)
    assert again.launches() == first.launches()
    again.launch()
    mtgp.synchronize()
    for g in (0, gens - 1):
        p = oracle.params(bits, mexp, g)
        want, _ = oracle.generate(p, oracle.init_state(p, 3 + g), 0, count)
        assert (buf.to_host(dt, count, g * count * eb) == want).all()
