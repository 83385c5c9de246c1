"""How pass programs reach the GPU: calls do not wait for earlier ones, and programs longer than
the ring they go through (several turns, and passes cut between rounds) leave the gates' state."""
import time

import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import random_state

pytestmark = pytest.mark.gpu


def test_calls_do_not_wait_for_earlier_ones(gpu):
    # 29 qubits: a call is some 10 ms on the GPU and some 2 on the host
    circ = circuits.brick(29, 3, seed=2)
    with pyqcs.Simulator(gpu, 29, seed=1) as sim:
        for _ in range(2):  # the first one is the warm-up
            sim.norm()
            t0 = time.perf_counter()
            for _ in range(4):
                sim.run(circ)
            queued = time.perf_counter() - t0
            sim.norm()
            total = time.perf_counter() - t0
    print("queued", queued, "total", total, flush=True)
    assert queued < 0.5 * total


# 12 qubits: one pass holds a call's whole program, and in the third call the ring ends in the
# middle of it; 13 and 17: many passes; the ring turns several times
@pytest.mark.parametrize("n,gates,calls", [(12, 4096, 5), (12, 300, 60), (13, 1000, 30), (17, 1500, 20)])
def test_programs_longer_than_the_ring(gpu, n, gates, calls):
    circ = circuits.random_all_gates(n, gates, seed=n, max_ctrls=2)
    psi = random_state(n, n)
    out = []
    for whole in (True, False):
        with pyqcs.Simulator(gpu, n, seed=3) as sim:
            sim.set_statevector(psi)
            for _ in range(calls):
                if whole:
                    sim.run(circ)
                else:
                    for op in circ:
                        sim.gate(*op)
            out.append(sim.statevector())
    # both sides round in FP64 at every gate, amplitudes of modulus <= 1
    assert np.max(np.abs(out[0] - out[1])) <= 16 * calls * gates * 2.0 ** -53 * np.max(np.abs(out[1]))
