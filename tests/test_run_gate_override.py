"""Simulator.run against a `gate` of a subclass's or an object's own: it is called for every gate."""
import types

import numpy as np
import pytest

import pyqcs
from pyqcs import circuits


class Counting(pyqcs.Simulator):
    def gate(self, name, *args, **kw):
        self.seen = getattr(self, "seen", []) + [name]
        super().gate(name, *args, **kw)


def check(lib):
    circ = circuits.random_all_gates(6, 30, seed=3)
    with pyqcs.Simulator(lib, 6) as plain, Counting(lib, 6) as sub, pyqcs.Simulator(lib, 6) as obj:
        seen = []

        def gate(self, name, *args, **kw):
            seen.append(name)
            pyqcs.Simulator.gate(self, name, *args, **kw)

        obj.gate = types.MethodType(gate, obj)
        for sim in (plain, sub, obj):
            sim.run(circ)
        assert sub.seen == seen == [op[0] for op in circ]
        want = plain.statevector()
        assert max(np.max(np.abs(s.statevector() - want)) for s in (sub, obj)) <= 16 * 30 * 2.0 ** -53


def test_oracle_run_calls_an_own_gate(oracle):
    check(oracle)


@pytest.mark.gpu
def test_gpu_run_calls_an_own_gate(gpu):
    check(gpu)
