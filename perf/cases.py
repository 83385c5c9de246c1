"""Performance cases: what users of the simulator run, through its public Python binding.

A case is one job: a circuit of one of the benchmark families on a state of `n` qubits in
one of the precision modes (0: complex128 per gate, 1: complex64 FP32 blocks, 2: complex128
FP64 blocks, 3: complex64 BF16x3 blocks), and what the job reads back.  Readouts of the
complex64 modes are returned as 32-bit values, the accuracy those states hold.

`prepare` makes what a program keeps from job to job (the allocated simulator and the
circuit with its angles, or the batch with its circuits added); `run` is one whole job from
a fresh state to its results on the host.
"""
import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "rqs-svg_amd"))

import pyqcs  # noqa: E402
from pyqcs import circuits  # noqa: E402


def listed():
    return [
        # a textbook-size circuit whose whole state comes back: the smallest calls, where
        # the cost of a call and a launch is everything
        {"name": "ghz6_state", "kind": "circuit", "circuit": "ghz", "n": 6, "depth": 4, "precision": 0, "read": "state"},
        # a variational evaluation of ordinary small size (all <Z_q> of a 13-qubit ansatz)
        {"name": "vqe13_expz", "kind": "circuit", "circuit": "variational", "n": 13, "depth": 6, "precision": 0, "read": "expz"},
        # the benchmark's 20-qubit job: H + CNOT chain, 20 layers of U3 + CZ, 1024 samples
        {"name": "ghz20_samples", "kind": "circuit", "circuit": "ghz", "n": 20, "depth": 20, "precision": 0, "read": "samples", "shots": 1024},
        # a QAOA evaluation on a state of ordinary size (diagonal two-qubit gates)
        {"name": "qaoa23_samples", "kind": "circuit", "circuit": "qaoa", "n": 23, "depth": 3, "precision": 0, "read": "samples", "shots": 8000},
        # the headline family at its full size: 16 GiB state, prefix and 4096 samples
        {"name": "brick30_samples", "kind": "circuit", "circuit": "brick", "n": 30, "depth": 3, "precision": 0, "read": "samples", "shots": 4096},
        # the per-shot path: a circuit, then every qubit measured in turn
        {"name": "brick27_measure", "kind": "measure", "circuit": "brick", "n": 27, "depth": 1, "precision": 0, "order": "up"},
        # a state loaded from the host, a few gates, and the state back to the host
        {"name": "load22_state", "kind": "load", "circuit": "random2q", "n": 22, "depth": 24, "precision": 0, "read": "state"},
        # the precision form on BF16x3 products, large state
        {"name": "vqe30_x3_expz", "kind": "circuit", "circuit": "variational", "n": 30, "depth": 4, "precision": 3, "read": "expz"},
        # the same form on FP32 MFMA at an ordinary, odd size: one step of a variational loop
        {"name": "vqe25_fp32_expz", "kind": "circuit", "circuit": "variational", "n": 25, "depth": 6, "precision": 1, "read": "expz"},
        # complex128 blocks on a phase-heavy circuit
        {"name": "qft27_f64_expz", "kind": "circuit", "circuit": "qft", "n": 27, "depth": 1, "precision": 2, "read": "expz"},
        # many small circuits in one call, FP32 block products (the default)
        {"name": "batch96", "kind": "batch", "count": 96, "nmin": 10, "nmax": 20, "dmin": 4, "dmax": 12, "precision": 1},
        # the same on BF16x3 block products, circuits that mostly fit LDS
        {"name": "batch256_small_x3", "kind": "batch", "count": 256, "nmin": 6, "nmax": 16, "dmin": 4, "dmax": 16, "precision": 3},
    ]


def draw(rng):
    kind = rng.choice(["circuit", "circuit", "circuit", "circuit", "measure", "load", "batch"])
    if kind == "batch":
        nmin = rng.randint(4, 14)
        nmax = nmin + rng.randint(2, 6)
        dmin = rng.randint(2, 6)
        return {"kind": "batch", "count": int(round(2 ** rng.uniform(3, 8))), "nmin": nmin, "nmax": nmax,
                "dmin": dmin, "dmax": dmin + rng.randint(1, 8), "precision": rng.choice([1, 3])}
    if kind == "load":
        return {"kind": "load", "circuit": rng.choice(["random2q", "qft", "brick"]), "n": rng.randint(8, 23),
                "depth": rng.randint(1, 24), "precision": rng.choice([0, 0, 2]), "read": "state"}
    if kind == "measure":
        return {"kind": "measure", "circuit": rng.choice(["brick", "ghz"]), "n": rng.randint(5, 27),
                "depth": rng.randint(1, 3), "precision": rng.choice([0, 0, 2, 3]), "order": rng.choice(["up", "down", "stride"])}
    precision = rng.choice([0, 0, 0, 1, 2, 3])
    # state sizes over their whole range; depths such that no job exceeds the largest listed one
    n = rng.randint(4, 28) if precision == 0 else rng.randint(14, 29)
    most = 6 if n >= 26 and precision == 0 else 12 if n >= 24 else 24
    family = rng.choice(["ghz", "brick", "variational", "qaoa", "qft", "random2q"])
    # <Z_q> is what a variational program reads (it is zero by symmetry after a GHZ chain or
    # a QAOA round); the others read samples or, where it is small enough, the state
    read = rng.choice(["samples", "state", "expz"]) if precision in (0, 2) else rng.choice(["state", "expz"])
    if read == "expz" and family in ("ghz", "qaoa"):
        family = "variational"
    if read == "state" and n > 22:
        n = rng.randint(14, 22)
    if read == "expz" and precision in (1, 3):
        family, most = "variational", 6
    case = {"kind": "circuit", "circuit": family, "n": n, "depth": rng.randint(1, most), "precision": precision, "read": read}
    if read == "samples":
        case["shots"] = int(round(2 ** rng.uniform(0, 13)))
    return case


def _circuit(case, seed):
    """The job's gates.  The seed sets every angle and random pairing; the QFT, which has
    neither, follows one random brick layer."""
    n, depth, s = case["n"], case["depth"], 1000003 * seed + 17
    kind = case["circuit"]
    if kind == "ghz":
        return circuits.ghz_u3_cz(n, depth, seed=s)
    if kind == "brick":
        return circuits.brick(n, depth, seed=s, mcx=2 if n >= 6 else 0)
    if kind == "variational":
        return circuits.variational(n, depth, seed=s)
    if kind == "qaoa":
        return circuits.qaoa_ring(n, depth, seed=s)
    if kind == "qft":
        return circuits.brick(n, 1, seed=s) + circuits.qft(n)
    if kind == "random2q":
        return circuits.random_two_qubit(n, depth * n, seed=s)
    raise ValueError(kind)


def _batch_circuits(case, seed):
    """Variational circuits whose sizes and depths are the case's own; the seed sets the angles."""
    sizes = circuits.variational_batch(case["count"], seed=case["count"] + 29, nmin=case["nmin"], nmax=case["nmax"], dmin=1, dmax=1)
    span, out = case["dmax"] - case["dmin"] + 1, []
    for i, (n, _) in enumerate(sizes):
        circ = circuits.variational(n, case["dmin"] + (7 * i) % span, seed=1000003 * seed + 31 * i)
        out.append((n, [(name, t[0], prm, c[0] if c else -1) for name, t, prm, c, _ in circ]))
    return out


def _input_state(n, seed):
    rng = np.random.default_rng([seed, n])
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    return psi / np.linalg.norm(psi)


def _measure_order(case):
    n = case["n"]
    if case["order"] == "up":
        return list(range(n))
    if case["order"] == "down":
        return list(range(n - 1, -1, -1))
    step = next(k for k in range(5, 5 + n) if math.gcd(k, n) == 1)
    return [(i * step) % n for i in range(n)]


def prepare(case, seed):
    lib = pyqcs.gpu_library()
    if case["kind"] == "batch":
        b = pyqcs.Batch(lib)
        for n, gates in _batch_circuits(case, seed):
            b.add(n, gates)
        if case["precision"] != 1:
            b.set_precision(case["precision"])
        return {"case": case, "batch": b}
    sim = pyqcs.Simulator(lib, case["n"], num_clbits=case["n"], seed=seed, precision=case["precision"])
    state = {"case": case, "seed": seed, "sim": sim, "circuit": _circuit(case, seed)}
    if case["kind"] == "load":
        state["psi"] = _input_state(case["n"], seed)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        z, _ = state["batch"].run()
        return np.concatenate(z).astype(np.float32)
    sim = state["sim"]
    if case["kind"] == "load":
        sim.set_statevector(state["psi"])
    else:
        sim.call("set_zero_state")
    sim.run(state["circuit"])
    if case["kind"] == "measure":
        sim.set_seed(state["seed"])
        for q in _measure_order(case):
            sim.measure_to_clbit(q, q)
        total = sim.probability_total()
        return {"bits": np.array(sim.clbits(), dtype=np.uint8),
                "total": np.array([total], dtype=np.float32 if case["precision"] in (1, 3) else np.float64)}
    if case["read"] == "samples":
        total = sim.probability_total()
        return {"total": total, "samples": sim.sample(case["shots"], seed=state["seed"])}
    if case["read"] == "expz":
        z = sim.expect_z()
        return z.astype(np.float32) if case["precision"] in (1, 3) else z
    psi = sim.statevector()
    return psi.astype(np.complex64) if case["precision"] in (1, 3) else psi


def _gate_flops(op):
    """Real operations per amplitude of the state: 14 for a dense 2x2 (two complex products
    and a sum), 6 for a phase, over the share that the controls and the phase's target leave."""
    name, _, _, ctrls, negctrls = op
    share = 0.5 ** (len(ctrls) + len(negctrls))
    if name in ("z", "p"):
        return 6 * share / 2
    if name in ("rz", "rzz"):
        return 6 * share
    if name in ("x", "swap"):
        return 0.0
    return 14 * share


def work(case):
    """The state written once and read once by what is read out, the readout itself, and
    the gates' arithmetic."""
    if case["kind"] == "batch":
        by = fl = 0.0
        for n, gates in _batch_circuits(case, 1):
            by += 2 * 8.0 * 2 ** n if n > 14 else 8.0 * n
            fl += 2.0 ** n * sum(_gate_flops((g[0], 0, 0, (0,) if g[3] >= 0 else (), ())) for g in gates)
        return {"bytes": by, "flops": fl}
    size = 8.0 if case["precision"] in (1, 3) else 16.0
    amps = 2.0 ** case["n"]
    by = 2 * size * amps
    if case["kind"] == "load":
        by += 2 * 16.0 * amps
    elif case.get("read") == "state":
        by += 16.0 * amps
    return {"bytes": by, "flops": amps * sum(_gate_flops(op) for op in _circuit(case, 1))}


# ---- the same results in plain 64-bit torch ----
def _matrix(name, p):
    r = 1 / math.sqrt(2)
    if name == "h":
        return [[r, r], [r, -r]]
    if name == "rx":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return [[c, -1j * s], [-1j * s, c]]
    if name == "ry":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return [[c, -s], [s, c]]
    if name == "u3":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        e = lambda a: complex(math.cos(a), math.sin(a))  # noqa: E731
        return [[c, -e(p[2]) * s], [e(p[1]) * s, e(p[1] + p[2]) * c]]
    if name == "x":
        return [[0, 1], [1, 0]]
    raise ValueError(name)


def _view(psi, n, qubits):
    """psi as a tensor with an axis of size 2 for each of `qubits`, and the axes, by qubit."""
    order = sorted(qubits, reverse=True)
    shape, axis, top = [], {}, n
    for q in order:
        shape += [1 << (top - q - 1), 2]
        axis[q] = len(shape) - 1
        top = q
    shape.append(1 << top)
    return psi.view(shape), axis


def _apply(psi, n, op):
    name, targets, params, ctrls, negctrls = op
    v, axis = _view(psi, n, list(targets) + list(ctrls) + list(negctrls))
    at = [slice(None)] * v.dim()
    for q in ctrls:
        at[axis[q]] = 1
    for q in negctrls:
        at[axis[q]] = 0

    def part(**bits):
        i = list(at)
        for q, b in bits.items():
            i[axis[int(q[1:])]] = b
        return v[tuple(i)]

    t = targets[0]
    if name in ("z", "p"):
        ph = -1.0 if name == "z" else complex(math.cos(params[0]), math.sin(params[0]))
        part(**{"q%d" % t: 1}).mul_(ph)
    elif name == "rz":
        a = params[0] / 2
        part(**{"q%d" % t: 0}).mul_(complex(math.cos(a), -math.sin(a)))
        part(**{"q%d" % t: 1}).mul_(complex(math.cos(a), math.sin(a)))
    elif name == "rzz":
        a, u = params[0] / 2, targets[1]
        for b in range(4):
            s = -1 if (b & 1) == (b >> 1) else 1
            part(**{"q%d" % t: b & 1, "q%d" % u: b >> 1}).mul_(complex(math.cos(a), s * math.sin(a)))
    elif name == "swap":
        u = targets[1]
        a, b = part(**{"q%d" % t: 0, "q%d" % u: 1}), part(**{"q%d" % t: 1, "q%d" % u: 0})
        keep = a.clone()
        a.copy_(b)
        b.copy_(keep)
    else:
        m = _matrix(name, params)
        a, b = part(**{"q%d" % t: 0}), part(**{"q%d" % t: 1})
        na = a * m[0][0]
        na.add_(b * m[0][1])
        b.mul_(m[1][1])
        b.add_(a * m[1][0])
        a.copy_(na)


def _simulate(n, ops, psi=None):
    if psi is None:
        psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
        psi[0] = 1
    for op in ops:
        _apply(psi, n, op)
    return psi


def _expz(psi, n):
    p = torch.view_as_real(psi).square().sum(-1)
    out = []
    for q in range(n):
        v = p.view(-1, 2, 1 << q).sum((0, 2))
        out.append(float(v[0] - v[1]))
    return out


def exact(case, seed):
    if case["kind"] == "measure":
        return None  # random outcomes and what they leave of the state
    if case["kind"] == "batch":
        if sum(2.0 ** n * len(g) for n, g in _batch_circuits(case, seed)) > 4e11:
            return None
        z = []
        for n, gates in _batch_circuits(case, seed):
            z += _expz(_simulate(n, circuits.batch_to_circuit(gates)), n)
        return torch.tensor(z, dtype=torch.float64)
    n, ops = case["n"], _circuit(case, seed)
    if 2.0 ** n * len(ops) > 6e11:
        return None
    start = torch.from_numpy(_input_state(n, seed)).cuda() if case["kind"] == "load" else None
    psi = _simulate(n, ops, start)
    if case["read"] == "state":
        return psi
    if case["read"] == "expz":
        return torch.tensor(_expz(psi, n), dtype=torch.float64)
    return {"total": float(torch.view_as_real(psi).square().sum()), "samples": None}
