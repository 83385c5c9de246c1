"""Which gates of a list run as passes and which as kernels of their own (the launches that the
profile counts), and that the state is the gates' either way."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import random_state

pytestmark = pytest.mark.gpu


def launches(sim, circ):
    sim.profile_reset()
    sim.profile(True)
    sim.run(circ)
    sim.norm()
    counts = {k: v["launches"] for k, v in sim.profile_get().items() if k != "reduce"}
    sim.profile(False)
    return counts


def mcx(n, controls, count, name="x"):
    rng = np.random.default_rng(n)
    out = []
    for _ in range(count):
        q = [int(x) for x in rng.permutation(n)[:controls + 1]]
        out.append((name, (q[0],), (), tuple(q[1:]), ()))
    return out


@pytest.mark.parametrize("n,controls,count,passes", [
    (10, 0, 2, False), (10, 0, 8, True), (20, 6, 2, False), (20, 6, 8, True),
    (22, 6, 2, False), (22, 6, 6, False), (22, 6, 16, True), (22, 0, 2, True), (24, 7, 6, False), (24, 0, 2, True)])
def test_short_lists(gpu, n, controls, count, passes):
    with pyqcs.Simulator(gpu, n, seed=1) as sim:
        got = launches(sim, mcx(n, controls, count))
    print("n", n, "controls", controls, "gates", count, got, flush=True)
    assert ("fused" in got) == passes and (got.get("pair", 0) == 0 if passes else got == {"pair": count})


# gates with more controls than a pass takes, alone, in a row, at both ends and between others
@pytest.mark.parametrize("n", [9, 12, 16, 20])
def test_gates_that_passes_do_not_take(gpu, oracle, n):
    wide = [("z", (n - 1,), (), tuple(range(n - 1)), ()), ("x", (0,), (), tuple(range(1, n)), ()),
            ("ry", (3,), (0.7,), tuple(q for q in range(n) if q not in (3, 5)), (5,))]
    layers = [circuits.brick(n, 2, seed=k, mcx=2) for k in range(3)]
    psi = random_state(n, n)
    for circ, singles in ((layers[0] + wide[:1] + layers[1], 1), (wide + layers[0] + wide[1:] + layers[1], 5),
                          (layers[0] + wide[2:] + layers[1][:1] + wide[:1] + layers[2], None), (wide, 3)):
        states = []
        for lib in (gpu, oracle):
            with pyqcs.Simulator(lib, n, seed=1) as sim:
                sim.set_statevector(psi)
                if lib is gpu:
                    got = launches(sim, circ)
                else:
                    sim.run(circ)
                states.append(sim.statevector())
        print("n", n, "gates", len(circ), got, flush=True)
        own = sum(v for k, v in got.items() if k != "fused")
        assert singles is None or own == singles
        assert (len(circ) == 3) == ("fused" not in got)
        assert np.max(np.abs(states[0] - states[1])) <= 16 * len(circ) * 2.0 ** -53 * np.max(np.abs(states[1]))
