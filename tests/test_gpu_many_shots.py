"""More outcomes than one fetch (65536): the two halves that they come through in turn, at their
edges, and the buffer kept for fewer and for more.  Outcomes are the oracle's, exactly."""
import numpy as np
import pytest

import pyqcs
from conftest import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 12])
def test_outcomes_of_many_fetches(gpu, oracle, n):
    most = 4 * 65536 + 3
    with pyqcs.Simulator(gpu, n, seed=1) as sim, pyqcs.Simulator(oracle, n, seed=1) as ref:
        for s in (sim, ref):
            s.set_statevector(random_state(n, n))
        want = ref.sample(most, seed=4)
        for shots in (65536, 65537, 3, 2 * 65536, 2 * 65536 + 1, 3 * 65536, most, 1, most):
            assert np.array_equal(sim.sample(shots, seed=4), want[:shots])
