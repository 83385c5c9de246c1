"""Circuit passes on the GPU: Simulator.run on a complex128 state against the same gates called
one by one (the per-gate kernels) and, at small sizes, against the oracle.  Both sides round
in FP64 at every gate: amplitudes of modulus <= 1 after g gates differ by at most a few
roundings each, so the bound is 16 g 2^-53 times the largest amplitude."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import random_state

pytestmark = pytest.mark.gpu


def both(gpu, n, circ, mapping=None):
    psi = random_state(n, n)
    out = []
    for whole in (True, False):
        with pyqcs.Simulator(gpu, n, mapping=mapping, seed=3) as sim:
            sim.set_statevector(psi)
            if whole:
                sim.run(circ)
            else:
                for op in circ:
                    sim.gate(*op)
            out.append(sim.statevector())
    return out


def bound(circ, psi):
    return 16 * len(circ) * 2.0 ** -53 * np.max(np.abs(psi))


# one-tile states around the smallest tile, the single-workgroup sizes, and the sizes where the
# tile grows; 24 and 25 qubits lie on both sides of the cached / non-temporal access switch
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 9, 10, 11, 12, 13, 14, 16, 17, 18, 19, 21])
def test_passes_match_gates(gpu, n):
    for seed in range(3 if n < 18 else 1):
        circ = circuits.random_all_gates(n, 120, seed=100 * n + seed, max_ctrls=min(4, n - 1)) if n > 1 else \
            [("h", (0,), (), (), ()), ("rz", (0,), (0.3,), (), ()), ("u3", (0,), (0.2, 0.7, 1.1), (), ()), ("y", (0,), (), (), ())]
        mapping = [int(q) for q in np.random.default_rng(seed).permutation(n)] if seed == 1 else None
        print("n", n, "seed", seed, flush=True)
        a, b = both(gpu, n, circ, mapping)
        assert np.max(np.abs(a - b)) <= bound(circ, b)


@pytest.mark.parametrize("n,family", [(24, "brick"), (25, "brick"), (20, "qft"), (20, "variational"), (19, "qaoa")])
def test_passes_match_gates_families(gpu, n, family):
    circ = {"brick": lambda: circuits.brick(n, 3, seed=5, mcx=3), "qft": lambda: circuits.qft(n),
            "variational": lambda: circuits.variational(n, 3, seed=6), "qaoa": lambda: circuits.qaoa_ring(n, 2, seed=7)}[family]()
    a, b = both(gpu, n, circ)
    assert np.max(np.abs(a - b)) <= bound(circ, b)


# programs longer than their staging area: several groups of passes, which start again at its
# beginning; and more gates than are planned together
@pytest.mark.parametrize("n,gates", [(13, 1500), (14, 5000), (20, 1200), (23, 400)])
def test_long_programs_match_gates(gpu, n, gates):
    circ = circuits.random_all_gates(n, gates, seed=gates, max_ctrls=2)
    a, b = both(gpu, n, circ)
    assert np.max(np.abs(a - b)) <= bound(circ, b)


def test_run_refuses_like_the_gates(gpu, oracle):
    # a refused gate in the middle: the ones before it are applied, the message is the gate's
    n = 7
    good = circuits.random_all_gates(n, 20, seed=8)
    for bad, text in ((("x", (9,), (), (), ()), "gate_x"), (("swap", (1, 1), (), (), ()), "more than once"), (("h", (1, 2), (), (), ()), "target")):
        states = []
        for lib in (gpu, oracle):
            with pyqcs.Simulator(lib, n, seed=1) as sim:
                with pytest.raises(pyqcs.QcsError, match=text):
                    sim.run(good + [bad] + good)
                states.append(sim.statevector())
        assert np.max(np.abs(states[0] - states[1])) <= 1e-13


def test_run_with_measured_qubits_and_profile(gpu, oracle):
    # measured qubits are implicit controls: such circuits go gate by gate
    n = 8
    c1, c2 = circuits.random_all_gates(n, 40, seed=11), circuits.random_all_gates(n, 40, seed=12)
    res = []
    for lib in (gpu, oracle):
        with pyqcs.Simulator(lib, n, seed=4) as sim:
            sim.run(c1)
            bits = [sim.measure(2), sim.measure(5)]
            sim.run(c2)
            sim.call("reset_measurement_state")
            sim.run(c1)
            res.append((bits, sim.statevector()))
    assert res[0][0] == res[1][0]
    assert np.max(np.abs(res[0][1] - res[1][1])) <= 1e-13


# The fused modes' default flushes: FP64 arithmetic, and for complex64 one rounding to FP32 of
# every amplitude per sweep (2^-24 of its modulus) and two more when the state is rescaled, which
# a unitary carries along unchanged: ||d|| <= (sweeps + 3) 2^-24 on a state of norm 1.
@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("n", [4, 5, 9, 10, 12, 13, 18, 19, 22, 24])
def test_fused_modes_run_as_passes(gpu, n, precision):
    circ = circuits.random_all_gates(n, 150, seed=n, max_ctrls=3 if n > 5 else 1) if n < 22 else circuits.brick(n, 3, seed=n, mcx=3)
    psi = random_state(n, n)
    with pyqcs.Simulator(gpu, n) as plain, pyqcs.Simulator(gpu, n, precision=precision) as fused:
        for sim in (plain, fused):
            sim.set_statevector(psi)
        for op in circ:
            plain.gate(*op)
        fused.run(circ)
        gates, sweeps = fused.fusion_stats()  # flushes
        d = np.linalg.norm(plain.statevector() - fused.statevector())
    print("n", n, "precision", precision, "sweeps", sweeps, "||d||", d, flush=True)
    assert gates == len(circ) and sweeps < len(circ)
    assert d <= (sweeps + 3) * 2.0 ** -24 if precision == 1 else d <= 16 * len(circ) * 2.0 ** -53


@pytest.mark.parametrize("precision,m", [(1, 13), (2, 12)])
def test_fused_modes_asked_for_stages(gpu, precision, m):
    # a stage size or a fixed plan turns passes off, also after a flush that ran as passes: the
    # stages' sweep count is that of a simulator that never ran a pass
    n = 17
    circ = circuits.brick(n, 6, seed=4, mcx=2)
    counts, states = [], []
    for before, plan in ((False, False), (True, False), (True, True)):
        with pyqcs.Simulator(gpu, n, precision=precision, stage_bits=None if before else 13) as sim:
            if before:
                sim.run(circ)
                sim.call("set_zero_state")
                sim.fusion_stats()
                sim.set_plan(m, 3 if precision == 2 else 5, tiles=2) if plan else sim.set_stage_bits(13)
            g0, s0 = sim.fusion_stats()
            sim.run(circ)
            g1, s1 = sim.fusion_stats()
            counts.append((g1 - g0, s1 - s0))
            states.append(sim.statevector())
    assert counts[0] == counts[1] == counts[2] and counts[0][0] == len(circ)
    assert np.array_equal(states[0], states[1]) and np.array_equal(states[0], states[2])


# Batches with no tuning set run as passes: the circuits of up to 12 qubits never leave FP64; a
# larger one is rounded to FP32 after every pass but the last (2^-24 of each modulus, carried
# along unchanged), and |d<Z>| <= 2 ||d|| + ||d||^2.  Together, alone, replayed and launched
# without the graph the circuits give the same bits.
@pytest.mark.parametrize("mode", [1, 3])
def test_batch_as_passes(gpu, oracle, mode):
    work = []
    for n in list(range(1, 15)) + ([15, 16, 17, 19] if mode == 1 else []):
        for depth in (1, 5) if n < 17 else (3,):
            work.append((n, circuits.variational_batch(1, seed=100 * n + depth, nmin=n, nmax=n, dmin=depth, dmax=depth)[0][1]))
    work.append((9, [("h", 3, (), -1), ("z", 3, (), 8), ("t", 0, (), -1), ("sx", 8, (), 0), ("u3", 5, (0.4, 1.0, 2.0), 2)]))
    work.append((13, [("y", 12, (), -1), ("p", 12, (0.3,), 0), ("x", 0, (), 12)]))  # one kind of gate a tile
    ref, whole = pyqcs.Batch(oracle), pyqcs.Batch(gpu)
    for n, g in work:
        ref.add(n, g)
        whole.add(n, g)
    whole.set_precision(mode)
    want, _ = ref.run()
    got, _ = whole.run()
    for again, _ in (whole.run(), whole.run_direct(), whole.run()):
        assert all(np.array_equal(x, y) for x, y in zip(got, again))
    for (n, g), z, w in zip(work, got, want):
        with_alone = pyqcs.Batch(gpu)
        with_alone.add(n, g)
        with_alone.set_precision(mode)
        alone, _ = with_alone.run()
        rounded = with_alone.traffic()["hbm_bytes"] / (16.0 * 2 ** n)
        d = rounded * 2.0 ** -24
        print("n", n, "gates", len(g), "roundings", rounded, "max|d<Z>|", np.max(np.abs(z - w)), flush=True)
        assert rounded == 0 if n <= 12 else rounded < len(g)
        assert np.max(np.abs(z - w)) <= 2 * d + d * d + 1e-13
        assert np.array_equal(alone[0], z)
        with_alone.close()
    whole.close()
    ref.close()
