"""What preparing a batch keeps on the host: the matrices of its stages and blocks are composed on the
device, and the host holds none of them meanwhile."""
import os
import threading
import time

import numpy as np
import pytest

import pyqcs

pytestmark = pytest.mark.gpu


def resident():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[1]) * os.sysconf("SC_PAGE_SIZE")


def work(count, gates):
    # pairs at random: hardly two of them share a block of 4 or 5 qubits
    rng = np.random.default_rng(count)
    circs = []
    for _ in range(count):
        pairs = [rng.permutation(15)[:2] for _ in range(gates)]
        circs.append([("ry", int(a), (0.3 + i,), int(b)) for i, (a, b) in enumerate(pairs)])
    return circs


def test_matrices_stay_on_the_device(gpu):
    def run(circs):
        b = pyqcs.Batch(gpu)
        for g in circs:
            b.add(15, g)
        b.set_precision(3)
        before, most, done = resident(), [0], threading.Event()

        def watch():
            while not done.is_set():
                most[0] = max(most[0], resident())
                time.sleep(0.0005)

        t = threading.Thread(target=watch)
        t.start()
        b.run()
        done.set()
        t.join()
        b.close()
        return most[0] - before

    run(work(2, 20))
    # The matrices take 16 KiB a block of 5 qubits, with 4 or 5 of these 51200 gates each: some
    # 180 MiB.  What the host does keep, about 100 bytes a gate, is below 20 MiB with its growth.
    grown = run(work(64, 800))
    print(f"the host's memory grew by {grown >> 20} MiB", flush=True)
    assert grown < 64 << 20
