"""Angles that are no number (NaN, infinity), among gates that a list would run as passes: only
the amplitudes that such a gate touches are lost, as where every gate is called by itself, which
is also what the oracle leaves."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import random_state

pytestmark = pytest.mark.gpu

N = 7


def bad(angle):
    return [("p", (2,), (angle,), (), ()), ("p", (1,), (angle,), (4,), (0,)), ("u3", (3,), (0.1, angle, 0.2), (5,), ()), ("rx", (6,), (angle,), (0, 1), ())]


@pytest.mark.parametrize("angle", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("which", range(4))
def test_lost_amplitudes_are_the_gates(gpu, oracle, angle, which):
    # diagonal gates around it: what is lost does not spread
    around = [g for g in circuits.random_all_gates(N, 300, seed=5, max_ctrls=2) if g[0] in ("z", "s", "t", "sdg", "tdg", "u1", "p", "rz", "rzz")]
    assert len(around) > 20
    circ = around[:10] + [bad(angle)[which]] + around[10:]
    psi = random_state(N, 1)
    got = []
    for lib, whole in ((gpu, True), (gpu, False), (oracle, False)):
        with pyqcs.Simulator(lib, N, seed=1) as sim:
            sim.set_statevector(psi)
            if whole:
                sim.run(circ)
            else:
                for op in circ:
                    sim.gate(*op)
            got.append(sim.statevector())
    lost = [np.isnan(s.real) | np.isnan(s.imag) for s in got]
    print(angle, which, "lost", [int(x.sum()) for x in lost], flush=True)
    assert 0 < lost[2].sum() < 1 << N
    assert (lost[0] == lost[1]).all() and (lost[1] == lost[2]).all()
    kept = ~lost[2]
    assert np.max(np.abs(got[0][kept] - got[2][kept])) <= 16 * len(circ) * 2.0 ** -53


@pytest.mark.parametrize("n", [4, 13])
def test_batches_with_such_an_angle(gpu, oracle, n):
    # the other circuits of the batch are not touched by it
    work = []
    for k in range(4):
        gates = [(nm, t[0], prm, c[0] if c else -1) for nm, t, prm, c, _ in circuits.variational(n, 2, seed=k)]
        work.append(gates[:5] + [("p", 1, (float("nan"),), 0)] + gates[5:] if k == 2 else gates)
    z = []
    for lib in (gpu, oracle):
        b = pyqcs.Batch(lib)
        for gates in work:
            b.add(n, gates)
        z.append(b.run()[0])
        b.close()
    assert np.isnan(z[1][2]).any()
    for k in (0, 1, 3):
        assert np.max(np.abs(z[0][k] - z[1][k])) <= 1e-5  # larger states round to FP32 a few times
    assert (np.isnan(z[0][2]) == np.isnan(z[1][2])).all()
