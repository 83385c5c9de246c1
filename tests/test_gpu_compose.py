"""Block matrices composed on the device, through the fused modes' blocks and stages: gates of no to
four targets, with controls inside the block and out, alone in a block and in long runs, and the
product tables of diagonal gates (also of gates that cancel to a diagonal), against the oracle.
Tolerances are those of the fused modes' products (FP32, and BF16x3 at about 2^-17 a factor)."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits
from conftest import fidelity, random_state

pytestmark = pytest.mark.gpu

FID_TOL, AMP_TOL = 1e-6, 1e-5


def check(gpu, oracle, n, circ, **how):
    psi = random_state(n, n)
    out = []
    for lib, kw in ((gpu, how), (oracle, {})):
        with pyqcs.Simulator(lib, n, **kw) as sim:
            sim.set_statevector(psi)
            sim.run(circ)
            out.append(sim.statevector())
    assert fidelity(out[0], out[1]) >= 1 - FID_TOL and np.max(np.abs(out[0] - out[1])) <= AMP_TOL


@pytest.mark.parametrize("precision,stage_bits", [(3, None), (1, 0), (1, 11)])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
def test_blocks_of_every_gate(gpu, oracle, k, precision, stage_bits):
    for n in (4, 5, 6, 9, 15) if k >= 4 else (4, 6):
        print("n", n, "k", k, "precision", precision, flush=True)
        circ = circuits.random_all_gates(n, 60, seed=10 * n + k, max_ctrls=min(3, n - 1))
        check(gpu, oracle, n, circ, precision=precision, block_qubits=k, stage_bits=stage_bits)


@pytest.mark.parametrize("gates", [1, 31, 32, 33, 200])
def test_runs_in_one_block(gpu, oracle, gates):
    # around the number of gates taken to LDS at a time, among them ones of 256 coefficients
    rng = np.random.default_rng(gates)
    circ = []
    for i in range(gates):
        q = [int(x) for x in rng.permutation(5)]
        circ.append([("ry", (q[0],), (rng.uniform(-3, 3),), (), ()), ("rcccx", tuple(q[:4]), (), (), ()), ("rzx", (q[1], q[2]), (0.4,), (q[0],), (q[3],)),
                     ("global_phase", (), (0.3,), (q[4],), ()), ("rccx", tuple(q[:3]), (), (), (q[4],))][i % 5])
    check(gpu, oracle, 8, circ, precision=3)


@pytest.mark.parametrize("precision", [1, 3])
def test_diagonal_tails(gpu, oracle, precision):
    # a stage that ends in diagonal gates, one of diagonal gates only, and pairs that cancel
    n = 17
    dense = [("ry", (q,), (0.3 + q,), (), ()) for q in range(6)]
    diag = [("p", (q,), (0.2 * q + 0.1,), (q + 1,), ()) for q in range(6)] + [("rzz", (2, 5), (0.7,), (), ()), ("t", (3,), (), (), (4,)), ("rz", (1,), (0.5,), (), ())]
    cancel = [("h", (7,), (), (), ()), ("h", (7,), (), (), ()), ("x", (8,), (), (7,), ()), ("x", (8,), (), (7,), ())]
    for circ in (dense + diag, diag, diag + cancel, cancel + diag + dense):
        check(gpu, oracle, n, circ, precision=precision, stage_bits=13)
