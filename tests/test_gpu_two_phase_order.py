"""Two-phase launches: every blocked jump first, then each phase's generation
in a launch of its own, over plans switched on after they were built, rebased
in between, relaunched, captured and switched back.  Whole numbers: every
comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("specs,count", [([(32, 11213, 0)] * 3, 400000), ([(64, 23209, 2), (64, 23209, 9)], 300001),
                                         ([(32, 44497, 1), (64, 44497, 3), (32, 11213, 8)], 500009)])
def test_jumps_then_the_generation_of_each_phase(mtgp, oracle, specs, count):
    print("two-phase order: %s" % (specs,), flush=True)
    gs = mtgp.GenSet(specs)
    gs.init_seed([41 + g for g in range(len(specs))])
    ps = [oracle.params(*s) for s in specs]
    ws = [oracle.init_state(p, 41 + g) for g, p in enumerate(ps)]
    bufs = [mtgp.DeviceBuffer(count * s[0] // 8) for s in specs]
    with mtgp.tuning(two_size_rho=1e9):
        plan = gs.plan([(g, 0, count, 0, b) for g, b in enumerate(bufs)])
    serial = plan.stats()["launches"]
    classes = len({(L["bits"], L["cls"]) for L in plan.launches()})
    assert serial == 3 * classes  # products, folds and generation of each class
    stream = mtgp.Stream()

    def check(launch):
        launch()
        stream.synchronize()
        for g, b in enumerate(bufs):
            want, _ = oracle.generate(ps[g], ws[g], 0, count)
            assert (b.to_host(want.dtype, count) == want).all(), g
            b.from_host(np.full(want.nbytes, 0x5A, np.uint8))

    def advance():
        plan.commit()
        plan.rebase(stream)
        for g in range(len(specs)):
            _, ws[g] = oracle.generate(ps[g], ws[g], 0, count)

    check(lambda: plan.launch(stream))
    advance()
    assert plan.set_overlap(True)
    assert plan.stats()["launches"] == serial + classes  # generation in each phase
    for _ in range(2):
        check(lambda: plan.launch(stream))
        check(lambda: plan.launch(stream))
        advance()
    plan.capture(stream)
    for _ in range(2):
        check(lambda: plan.launch_graph(stream))
        plan.launch(stream)
        advance()
    plan.set_overlap(False)
    assert plan.stats()["launches"] == serial
    check(lambda: plan.launch(stream))
