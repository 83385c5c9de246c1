"""How far passes and gates called one by one are from the exact state: 80-bit amplitudes and
angles, four circuit families.  Both err by a few roundings a gate, so over several circuits
their errors (root of the summed squares) are about the same; the bound leaves a quarter."""
import numpy as np
import pytest

import pyqcs
from pyqcs import circuits

pytestmark = pytest.mark.gpu

F, C = np.longdouble, np.clongdouble


def exp(a):
    return C(np.cos(a) + 1j * np.sin(a))


def matrix(name, p):
    p = [F(v) for v in p]
    if name in ("x", "z", "h"):
        r = 1 / np.sqrt(F(2))
        return {"x": [[0, 1], [1, 0]], "z": [[1, 0], [0, -1]], "h": [[r, r], [r, -r]]}[name]
    if name == "p":
        return [[1, 0], [0, exp(p[0])]]
    if name == "rz":
        return [[exp(-p[0] / 2), 0], [0, exp(p[0] / 2)]]
    c, s = np.cos(p[0] / 2), np.sin(p[0] / 2)
    if name == "rx":
        return [[c, -1j * s], [-1j * s, c]]
    if name == "ry":
        return [[c, -s], [s, c]]
    assert name == "u3"
    return [[c, -exp(p[2]) * s], [exp(p[1]) * s, exp(p[1] + p[2]) * c]]


def exact(n, circ):
    psi = np.zeros(1 << n, dtype=C)
    psi[0] = 1
    i = np.arange(1 << n)
    for name, targets, params, ctrls, negctrls in circ:
        on = np.ones(1 << n, dtype=bool)
        for q in ctrls:
            on &= (i >> q) & 1 == 1
        for q in negctrls:
            on &= (i >> q) & 1 == 0
        if name == "rzz":
            odd = ((i >> targets[0]) ^ (i >> targets[1])) & 1 == 1
            psi = np.where(on, psi * np.where(odd, exp(F(params[0]) / 2), exp(-F(params[0]) / 2)), psi)
            continue
        bit = 1 << targets[0]
        m = matrix(name, params)
        lo = i[on & (i & bit == 0)]
        a, b = psi[lo], psi[lo | bit]
        psi[lo], psi[lo | bit] = m[0][0] * a + m[0][1] * b, m[1][0] * a + m[1][1] * b
    return psi


@pytest.mark.parametrize("n", [6, 10, 13])
@pytest.mark.parametrize("family", ["ghz", "brick", "variational", "qaoa"])
def test_error_of_passes_and_of_gates(gpu, n, family):
    make = {"ghz": lambda s: circuits.ghz_u3_cz(n, 6, seed=s), "brick": lambda s: circuits.brick(n, 6, seed=s, mcx=2),
            "variational": lambda s: circuits.variational(n, 4, seed=s), "qaoa": lambda s: circuits.qaoa_ring(n, 4, seed=s)}[family]
    square = [0.0, 0.0]
    for seed in range(6):
        circ = make(seed)
        want = exact(n, circ)
        for k, whole in enumerate((True, False)):
            with pyqcs.Simulator(gpu, n, seed=1) as sim:
                if whole:
                    sim.run(circ)
                else:
                    for op in circ:
                        sim.gate(*op)
                d = sim.statevector().astype(C) - want
            square[k] += float(np.sum(d.real ** 2 + d.imag ** 2))
    passes, gates = (float(np.sqrt(v)) for v in square)
    print(family, n, "passes", passes, "gates", gates, "ratio", passes / gates, flush=True)
    assert passes <= 1.25 * gates
