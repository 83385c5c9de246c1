"""Measured qubits whose zeros are no longer where their physical positions say: a later collapse
may not leave any part of the state alone then.  Against the oracle, which always writes the whole
half: results, amplitudes (one FP64 rounding at most: the collapses only zero) and exact zeros."""
import glob
import os
import threading
import time

import numpy as np
import pytest

import pyqcs
from conftest import random_state

pytestmark = pytest.mark.gpu


# reinitialize_mapping gives the qubits other positions and moves no data; window: the measured
# qubit was swapped in from above the local ones, which also leaves a mapping to go back from
@pytest.mark.parametrize("n,first,window", [(8, 5, None), (8, 7, 6), (9, 7, None), (13, 8, None)])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_measure_after_reinitialize_mapping(gpu, oracle, n, first, window, precision):
    if window and precision:
        pytest.skip("the window is a mode of the per-gate state")
    res = []
    for lib, prec in ((gpu, precision), (oracle, 0)):
        with pyqcs.Simulator(lib, n, seed=5, precision=prec) as sim:
            sim.set_statevector(random_state(n, n))
            if window:
                sim.set_local_qubits(window)
                sim.gate("h", (n - 1,))
            bits = [sim.measure(first)]
            if not window:
                sim.permute(list(range(n))[::-1])
            sim.call("reinitialize_mapping")
            bits += [sim.measure(q) for q in [q for q in range(n) if q != first][1::3]]
            res.append((bits, sim.statevector()))
    (g, a), (o, b) = res
    print("n", n, "precision", precision, "bits", g, o, flush=True)
    assert g == o and ((a == 0) == (b == 0)).all()
    assert np.max(np.abs(a - b)) <= (2.0 ** -52 if precision != 1 else 2.0 ** -23)


def test_measure_after_a_load_that_fails_midway(gpu, tmp_path):
    # The file is cut once the load has read into it: it throws with part of the state replaced,
    # and the measured qubit (still listed as measured) is non-zero on both sides there.
    n = 25  # 512 MiB, read 32 MiB at a time
    path = tmp_path / "state.bin"
    block = np.full(1 << 21, 2.0 ** (-n / 2), dtype=np.complex128)
    with open(path, "wb") as f:
        for _ in range(1 << (n - 21)):
            f.write(block)

    def position():
        for fd in glob.glob("/proc/self/fd/*"):
            try:
                if os.readlink(fd) == str(path):
                    with open(fd.replace("/fd/", "/fdinfo/")) as f:
                        return int(f.readline().split()[1])
            except OSError:
                pass
        return 0

    stop = threading.Event()

    def cut():
        size = path.stat().st_size
        while not stop.is_set():
            if 3 * block.nbytes <= position() < size:
                os.truncate(path, 4 * block.nbytes)
                return
            time.sleep(1e-4)

    with pyqcs.Simulator(gpu, n, seed=5) as sim:
        sim.call("set_flat_state")
        sim.measure(5)
        t = threading.Thread(target=cut)
        t.start()
        try:
            with pytest.raises(pyqcs.QcsError, match="fread"):
                sim.load(path)
        finally:
            stop.set()
            t.join()
        bit = sim.measure(6)
        psi = sim.statevector()
    rejected = psi.reshape(-1, 2, 1 << 6)[:, 1 - bit]
    assert np.count_nonzero(psi) > 0 and not rejected.any()
