"""Measurements after measurements on the GPU against the oracle: a collapse leaves the part of the
state alone that earlier ones have zeroed, so sequences of measurements, gates and new states in
every order of qubits have to give the oracle's results, its amplitudes and exactly its zeros."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import random_state

pytestmark = pytest.mark.gpu


def play(lib, n, order, precision, mapping, steps):
    """Measures order[:len(order) // 2], does the steps, measures the rest."""
    out = []
    with pyqcs.Simulator(lib, n, seed=7, precision=precision, mapping=mapping, num_clbits=n) as sim:
        sim.set_statevector(random_state(n, n))
        half = len(order) // 2
        out.append([sim.measure_to_clbit(q, q) for q in order[:half]])
        out.append(sim.statevector())
        for step in steps:
            if step == "gates":  # measured qubits as targets, controls and neither
                a, b, c = order[0], order[half - 1], order[-1]
                for g in [("h", (c,), (), (), ()), ("x", (a,), (), (), ()), ("u3", (c,), (0.3, 0.1, 0.2), (b,), ()), ("swap", (b, c), (), (), ()), ("ry", (b,), (0.7,), (), ())]:
                    sim.gate(*g)
            elif step == "random":  # a new state that keeps the measured qubits
                sim.call("set_random_state")
        out.append([sim.measure_to_clbit(q, q) for q in order[half:]])
        out.append(sim.statevector())
        out.append(sim.norm())
    return out


# sizes around the line rule's smallest state (8 qubits) and one of several reduction tiles
@pytest.mark.parametrize("n", [4, 7, 8, 9, 14])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_measurement_sequences(gpu, oracle, n, precision):
    up = list(range(n))
    for i, order in enumerate((up, up[::-1], up[::2] + up[1::2])):
        for steps in ((), ("gates",), ("random",)):
            mapping = [int(q) for q in np.random.default_rng(n).permutation(n)] if i == 2 else None
            print("n", n, "precision", precision, "order", i, steps, flush=True)
            g, o = play(gpu, n, order, precision, mapping, steps), play(oracle, n, order, 0, mapping, steps)
            tol = 1e-13 if precision != 1 else 1e-6  # FP64, or every amplitude rounded to FP32 a few times
            assert g[0] == o[0] and g[2] == o[2]
            unit = precision == 1 and steps == ("gates",)  # a flush of complex64 gates rescales to norm 1
            for a, b in ((g[1], o[1]), (g[3], o[3])):
                if unit:
                    a, b = a / np.linalg.norm(a), b / np.linalg.norm(b)
                assert np.max(np.abs(a - b)) <= tol * max(1.0, np.max(np.abs(b)))
                assert np.array_equal(a == 0, b == 0) or steps == ("gates",)  # gates: zeros by rounding
            assert unit or abs(g[4] - o[4]) <= tol * max(1.0, o[4])


# The qubits inside a line of 128 B and around half of it, before, between and after others that
# narrow the collapse, with and without the rescale.
@pytest.mark.parametrize("n", [7, 8, 10])
@pytest.mark.parametrize("renormalize", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
def test_collapse_within_lines(gpu, oracle, n, renormalize, precision):
    tol = 1e-13 if precision == 0 else 1e-6  # as above
    for order in ((0, 1, 2, 3, 4, 5), (4, 3, 2, 1, 0), (2, 5, 3, 0, 4), (3, 1, 2, 6)):
        res = []
        for lib, prec in ((gpu, precision), (oracle, 0)):
            with pyqcs.Simulator(lib, n, seed=11, precision=prec, num_clbits=n) as sim:
                sim.set_renormalize(renormalize)
                sim.set_statevector(random_state(n, n + 1))
                for q in order:
                    res.append((sim.measure_to_clbit(q, q), sim.statevector()))
        for (r, a), (s, b) in zip(res[:len(order)], res[len(order):]):
            assert r == s and np.array_equal(a == 0, b == 0)
            assert np.max(np.abs(a - b)) <= tol * max(1.0, np.max(np.abs(b)))


# Whole and partial blocks of 64 at the top level, one level and several; more shots than are
# fetched at a time; a state whose zeros make long runs of equal prefixes.  Outcomes are integers
# from FP64 sums in a fixed order: exactly the oracle's.
@pytest.mark.parametrize("n,shots", [(1, 5), (2, 100), (5, 64), (6, 65), (7, 1000), (11, 70000), (12, 1), (13, 3000), (18, 65537)])
def test_sampling_is_the_oracles(gpu, oracle, n, shots):
    psi = random_state(n, n)
    holes = np.where(np.arange(1 << n) % 7 < 5, 0.0, psi)
    states = [psi] + ([holes / np.linalg.norm(holes)] if n > 3 else [])
    for k, state in enumerate(states):
        res = []
        for lib in (gpu, oracle):
            with pyqcs.Simulator(lib, n, seed=1) as sim:
                sim.set_statevector(state)
                res.append((sim.sample(shots, seed=9 + k), sim.probability_total()))
                if lib is gpu:  # the buffer is kept: fewer shots, then as many again
                    assert np.array_equal(sim.sample(max(1, shots // 3), seed=9 + k), res[-1][0][:max(1, shots // 3)])
                    assert np.array_equal(sim.sample(shots, seed=9 + k), res[-1][0])
        assert res[0][1] == res[1][1] and np.array_equal(res[0][0], res[1][0])
