"""<Z> of one qubit alone (qcs_ext_expect_z with count 1, its own signed reduction): the bits that
the reduction of all qubits gives, whatever bit of the index the qubit is: inside a pair of
complex64 amplitudes, inside a tile, above it."""
import ctypes

import numpy as np
import pytest

import pyqcs
from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 4, 11, 13, 14, 18])
@pytest.mark.parametrize("precision", [0, 1])
def test_one_qubit_has_the_bits_of_all(gpu, oracle, n, precision):
    if precision and n < 4:
        pytest.skip("complex64 states have at least 4 qubits")
    psi = random_state(n, n)
    for place in range(n):
        mapping = [q for q in range(1, n)]
        mapping.insert(place, 0)  # physical bit `place` holds logical qubit 0
        with pyqcs.Simulator(gpu, n, mapping=mapping, seed=1, precision=precision) as sim, pyqcs.Simulator(oracle, n, mapping=mapping, seed=1) as ref:
            sim.set_statevector(psi)
            one = ctypes.c_double()
            sim._call(gpu.lib.qcs_ext_expect_z(sim.h, ctypes.addressof(one), 1), "expect_z")
            assert one.value == sim.expect_z()[0]
            if precision == 0:
                ref.set_statevector(psi)
                assert one.value == ref.expect_z()[0]
