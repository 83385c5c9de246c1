"""<Z_q> of every qubit from one read of the state (qcs_ext_expect_z): complex128 bit for bit
the oracle's canonical signed sums on the same state, complex64 within FP64 rounding of sums
over the simulator's own state.  Sizes: below, at and above a tile of 4096 units, several tiles
(one and two further levels), and every bit position of each level."""
import numpy as np
import pytest

import pyqcs
from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 11, 12, 13, 16, 20, 25])
def test_expect_z_complex128_bits(gpu, oracle, n):
    psi = random_state(n, 40 + n)
    mapping = [int(q) for q in np.random.default_rng(n).permutation(n)]
    z = []
    for lib in (gpu, oracle):
        with pyqcs.Simulator(lib, n, mapping=mapping, seed=1) as sim:
            sim.set_statevector(psi)
            z.append((sim.expect_z(), sim.norm()))
    assert np.array_equal(z[0][0], z[1][0])
    assert z[0][1] == z[1][1]


@pytest.mark.parametrize("n", [4, 5, 12, 13, 14, 18, 25, 26])
def test_expect_z_complex64(gpu, n):
    psi = random_state(n, 50 + n)
    with pyqcs.Simulator(gpu, n, seed=1, precision=1) as sim:
        sim.set_statevector(psi)
        z = sim.expect_z()
        own = sim.statevector()
    p = own.real ** 2 + own.imag ** 2
    for q in range(n):
        v = p.reshape(-1, 2, 1 << q)
        want = float(v[:, 0].sum() - v[:, 1].sum())
        # two FP64 sums of 2^n values adding to 1, pairwise trees on both sides: a few ulp of 1
        # per level
        assert abs(z[q] - want) <= 4 * n * 2.0 ** -53
