#!/usr/bin/env python3
"""Benchmark: 30-qubit complex128 brick circuit on one MI355X (plain method).

One step = zero state + 24 brick layers (U3 on all 30 qubits, CZ on even/odd neighbour
pairs alternating) with 4 three-control X gates (at least one operand among the top 6
qubits) + full-register probability reduction + 4096 seeded samples.  That is 1072 gate
calls on a 16 GiB state.  `value` is gates per second over the timed steps; the state is
resident in HBM throughout.

Also reported:
  roofline      -- the dominant kernel (the circuit pass, which applies the gates whose
                   targets lie in its tiles in one sweep of the state), its algorithmic
                   bytes per launch (2 * 16 B * amplitudes) over its average duration
                   from HIP events recorded around each launch on the simulator's stream
                   during the timed steps, against 8 TB/s;
  cpu_baseline  -- the oracle (the reference's plain method restated in C++/OpenMP) on the
                   host cores, on a bounded sample of the same workload;
  fused_c64     -- the precision form on the 32-qubit brick circuit of depth 32 (complex64
                   state, gates fused into k=5 blocks on FP32 MFMA; fused_c64_bf16x3 the
                   same on BF16x3 split-precision MFMA) against the plain FP64
                   method on the same GPU: time of each, speedup, and fidelity /
                   max |d amp| of the fused state against the FP64 state (both resident in
                   HBM, compared on the GPU in FP64);
  batch         -- 512 variational circuits of 12-22 qubits in one autotuned hipGraph
                   launch against a per-circuit plain-method loop, with max |d<Z>|;
  planner       -- the learned fusion planner: launch timings recorded at 26-32 qubits,
                   cost-model MLP trained on the GPU, then a 33-qubit QFT and a 33-qubit
                   brick circuit of depth 40 (complex128 fused): the greedy fusion
                   fallback, the plan the model picks, and the stage heuristic.
"""
import argparse
import json
import os
import pathlib
import sys
import time

import numpy as np

REPO = pathlib.Path(__file__).resolve().parent
sys.path.insert(0, str(REPO / "rqs-svg_amd"))

import pyqcs  # noqa: E402
from pyqcs import circuits  # noqa: E402

HBM_PEAK = 8.0e12
CIRCUIT_SEED = 20250101
SAMPLE_SEED = 4242


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def brief(x):
    """The result with its numbers to 6 digits (those near 1, the fidelities, to 12), so that the
    line stays short of 16000 characters, the length that is kept of a run's output."""
    if isinstance(x, dict):
        return {k: brief(v) for k, v in x.items()}
    if isinstance(x, (list, tuple)):
        return [brief(v) for v in x]
    if isinstance(x, float):
        return float(f"{x:.12g}" if abs(x - 1) < 1e-3 else f"{x:.6g}")
    return x


def traffic_from_profiles():
    """HBM bytes per pass measured with rocprofv3 PMC counters, if committed."""
    f = REPO / "profiles" / "pass_kernel_brick30_traffic.json"
    if not f.exists():
        return None
    try:
        return json.loads(f.read_text()).get("hbm_bytes_per_launch")
    except Exception:
        return None


def cpu_baseline(n, circ, budget_s=20.0):
    """Time the oracle on the first gates of the same circuit (30 qubits, host cores)."""
    lib = pyqcs.oracle_library()
    cores = len(os.sched_getaffinity(0))
    cores = min(cores, int(os.environ.get("OMP_NUM_THREADS", cores)))
    t_alloc = time.perf_counter()
    sim = pyqcs.Simulator(lib, n, seed=1)
    t0 = time.perf_counter()
    done = 0
    for op in circ:
        sim.gate(*op)
        done += 1
        if time.perf_counter() - t0 > budget_s:
            break
    dt = time.perf_counter() - t0
    sim.close()
    log(f"cpu baseline: {done} gates in {dt:.2f}s (alloc+init {t0 - t_alloc:.2f}s)")
    return {
        "value": done / dt,
        "unit": "gates/s",
        "cores": cores,
        "kind": "port",
        "sample": f"first {done} gates of the same 30-qubit brick circuit (U3 on q0.., then CZ), "
                  f"complex128, oracle/qcs_oracle.cpp with OpenMP, {budget_s:.0f}s budget",
    }


def small_leg(n=20, layers=20, shots=1024):
    """The reference's CPU-runnable case on one GPU against the oracle on the host cores:
    20 qubits complex128, H then a CNOT chain (GHZ), 20 layers of U3 on every qubit and CZ
    on a random perfect matching, 1024 samples.  Both run the same API calls; the
    timed region is the circuit from |0...0> plus the sampling, states allocated."""
    circ = circuits.ghz_u3_cz(n, layers, seed=CIRCUIT_SEED + 11)
    res = {}
    for name, lib in (("gpu", pyqcs.gpu_library()), ("cpu", pyqcs.oracle_library())):
        with pyqcs.Simulator(lib, n, seed=1) as s:
            s.run(circ[:n])  # first launches / first touch
            best = None
            for _ in range(3 if name == "gpu" else 1):
                s.call("set_zero_state")
                s.norm()
                t0 = time.perf_counter()
                s.run(circ)
                smp = s.sample(shots, seed=SAMPLE_SEED)
                dt = time.perf_counter() - t0
                best = dt if best is None else min(best, dt)
            res[name] = (best, s.statevector(), smp)
    cores = len(os.sched_getaffinity(0))
    cores = min(cores, int(os.environ.get("OMP_NUM_THREADS", cores)))
    (tg, psi_g, s_g), (tc, psi_c, s_c) = res["gpu"], res["cpu"]
    diff = float(np.max(np.abs(psi_g - psi_c)))
    same = int(np.sum(s_g == s_c))
    log(f"small leg: {n} q c128, {len(circ)} gates + {shots} samples: GPU {tg * 1e3:.1f} ms, "
        f"CPU oracle {tc * 1e3:.1f} ms on {cores} cores ({tc / tg:.1f}x); max|d amp| {diff:.1e}, "
        f"{same}/{shots} samples identical")
    return {"config": f"{n} qubits complex128: H + CNOT chain, {layers} layers U3 on all + CZ on a "
                      f"random matching, {shots} samples (plain method)",
            "gates": len(circ), "shots": shots, "gpu_s": tg, "gpu_gates_per_s": len(circ) / tg,
            "cpu_oracle_s": tc, "cpu_cores": cores, "gpu_vs_cpu": tc / tg,
            "max_abs_diff_amp": diff, "samples_identical": same}


FUSED_VARIANTS = (
    # (result key, precision mode, stage tile bits)
    ("fused_c64", 1, 13),
    ("fused_c64_bf16x3", 3, 13),
    ("fused_c64_bf16x3_per_block", 3, 0),
)


def fused_leg(n, depth, k, shots, variants=FUSED_VARIANTS):
    """Config: 32 qubits, brick depth 32; fused complex64 vs plain complex128 on one GPU.
    Precision mode 1 runs the blocks on FP32 MFMA, mode 3 on BF16x3 split-precision MFMA;
    stage tile bits 13 apply several blocks per sweep on LDS-resident tiles of 2^13
    amplitudes, 0 launches one sweep per block."""
    lib = pyqcs.gpu_library()
    circ = circuits.brick(n, depth, seed=CIRCUIT_SEED + 3)
    warm = circuits.brick(n, 1, seed=1)[: n + 2]
    plain = pyqcs.Simulator(lib, n, seed=1)
    plain.run(warm)
    plain.call("set_zero_state")
    plain.norm()
    t0 = time.perf_counter()
    plain.run(circ)
    plain.probability_total()
    t_plain = time.perf_counter() - t0
    log(f"fused leg: plain c128 {t_plain:.3f}s")
    out = {}
    for key, mode, stage_bits in variants:
        math_name = {1: "FP32 MFMA", 3: "BF16x3 split-precision MFMA"}[mode]
        how = f"stages on 2^{stage_bits}-amplitude LDS tiles" if stage_bits else "one sweep per block"
        res = {"config": f"brick{n}: {n} qubits, {depth} brick layers (U3 all + CZ even/odd), "
                         f"{len(circ)} gates, {shots} samples; complex64 state, k={k} blocks on "
                         f"{math_name}, {how}",
               "gates": len(circ), "block_qubits": k, "precision_mode": mode, "stage_bits": stage_bits}
        fused = pyqcs.Simulator(lib, n, seed=1, precision=mode, block_qubits=k, stage_bits=stage_bits)
        fused.run(warm)
        fused.call("set_zero_state")
        fused.norm()
        g0, b0 = fused.fusion_stats()
        fused.profile_reset()
        fused.profile(True)
        t0 = time.perf_counter()
        fused.run(circ)
        total = fused.probability_total()
        t_fused = time.perf_counter() - t0
        fused.profile(False)
        g1, b1 = fused.fusion_stats()
        blk = fused.profile_get().get("fused", {"launches": 1, "seconds": 1.0, "bytes": 0.0})
        ts = time.perf_counter()
        fused.sample(shots, seed=SAMPLE_SEED)
        t_sample = time.perf_counter() - ts
        ov, maxdiff = fused.overlap(plain)
        norm64, norm128 = fused.norm(), plain.norm()
        fid = abs(ov) ** 2 / (norm64 * norm128)
        raw = abs(ov) ** 2 / norm128  # unnormalised: a norm drift of the complex64 state counts
        stream = stage_bits == 13 and 22 <= n <= 33
        if stream:
            # the same flushes with one workgroup per tile in place of the streaming kernel
            # (bit-identical states; tests/test_gpu_fused.py checks the bits)
            fused.set_stage_stream(False)
            fused.call("set_zero_state")
            fused.norm()
            fused.profile_reset()
            fused.profile(True)
            t0 = time.perf_counter()
            fused.run(circ)
            fused.probability_total()
            t_tile = time.perf_counter() - t0
            fused.profile(False)
            tb = fused.profile_get().get("fused", {"launches": 1, "seconds": 1.0})
            waves = 2 if mode == 3 else 4  # waves per workgroup of k_stage on 2^13 tiles
            res["tile_per_workgroup"] = {"kernel": f"k_stage<{k}, {stage_bits}, {'true' if mode == 3 else 'false'}, {waves}>",
                                         "fused_c64_s": t_tile, "avg_ms": tb["seconds"] / tb["launches"] * 1e3,
                                         "streaming_speedup": t_tile / t_fused}
            log(f"fused leg: {key} with one workgroup per tile {t_tile:.3f}s ({t_tile / t_fused:.3f}x the streaming kernel's time)")
        fused.close()
        log(f"fused leg: {key} {t_fused:.3f}s ({b1 - b0} sweeps), fidelity {fid:.12f}, unnormalised "
            f"{raw:.12f}, |norm-1| {abs(norm64 - 1):.2e}, max|d| {maxdiff:.2e}")
        res.update({"plain_c128_s": t_plain, "fused_c64_s": t_fused, "speedup": t_plain / t_fused,
                    "sweeps": b1 - b0,
                    "fidelity": fid, "infidelity": 1 - fid, "overlap_unnormalised": raw,
                    "norm_deviation": abs(norm64 - 1), "max_abs_diff": maxdiff,
                    "probability_total": total, "sample_s": t_sample})
        # fused kernel: algorithmic bytes = one read and one write of the touched amplitudes
        # per launch (2 * 8 B * 2^n for a stage); each block costs 8 * 2^k flops per amplitude
        gbs = blk["bytes"] / blk["seconds"] / 1e9
        x3 = "true" if mode == 3 else "false"
        kern = (f"k_stage_stream<{k}, {stage_bits}, {x3}>" if stream else f"k_stage<{k}, {stage_bits}, {x3}>") if stage_bits \
            else f"k_block_lds<{k}, {x3}>"
        res["roofline"] = {"bound": "hbm", "kernel": kern,
                           "achieved": gbs, "peak": HBM_PEAK / 1e9, "unit": "GB/s",
                           "frac": gbs / (HBM_PEAK / 1e9), "launches": blk["launches"],
                           "avg_ms": blk["seconds"] / blk["launches"] * 1e3}
        log(f"fused leg: {kern} {gbs:.1f} GB/s over {blk['launches']} launches")
        out[key] = res
    plain.close()
    return out


def qft_c64_leg(n=32, k=5, stage_bits=13):
    """A phase-heavy circuit in the precision form: the n-qubit QFT (H, controlled-phase
    ladders, closing swaps) as complex64 stages (FP32 and BF16x3 MFMA; stages whose blocks
    are all diagonal run as one phase-table pass) against the plain complex128 method.  The
    QFT acts on the state of one random brick layer (on |0...0> it would only make the
    uniform superposition); that preparation is not timed."""
    lib = pyqcs.gpu_library()
    circ = circuits.qft(n)
    warm = circuits.brick(n, 1, seed=1)[: n + 2]
    prep = circuits.brick(n, 1, seed=CIRCUIT_SEED + 9)
    plain = pyqcs.Simulator(lib, n, seed=1)
    plain.run(warm)
    plain.call("set_zero_state")
    plain.run(prep)
    plain.norm()
    t0 = time.perf_counter()
    plain.run(circ)
    plain.probability_total()
    t_plain = time.perf_counter() - t0
    out = {"config": f"qft{n}: {n}-qubit QFT ({len(circ)} gates), complex64 stages of k={k} blocks "
                     f"on 2^{stage_bits}-amplitude tiles vs plain complex128, on the state of one "
                     f"random brick layer",
           "gates": len(circ), "plain_c128_s": t_plain}
    for mode, key in ((3, "bf16x3"), (1, "fp32")):
        fused = pyqcs.Simulator(lib, n, seed=1, precision=mode, block_qubits=k, stage_bits=stage_bits)
        fused.run(warm)
        fused.call("set_zero_state")
        fused.run(prep)
        fused.norm()
        g0, b0 = fused.fusion_stats()
        t0 = time.perf_counter()
        fused.run(circ)
        fused.probability_total()
        dt = time.perf_counter() - t0
        g1, b1 = fused.fusion_stats()
        ov, maxdiff = fused.overlap(plain)
        norm64, norm128 = fused.norm(), plain.norm()
        fid = abs(ov) ** 2 / (norm64 * norm128)
        raw = abs(ov) ** 2 / norm128
        fused.close()
        log(f"qft leg: {key} {dt:.3f}s ({b1 - b0} sweeps) vs plain c128 {t_plain:.3f}s = {t_plain / dt:.1f}x, "
            f"fidelity {fid:.12f}, unnormalised {raw:.12f}, |norm-1| {abs(norm64 - 1):.2e}, max|d| {maxdiff:.2e}")
        out[key] = {"fused_c64_s": dt, "sweeps": b1 - b0, "speedup": t_plain / dt,
                    "fidelity": fid, "infidelity": 1 - fid, "overlap_unnormalised": raw,
                    "norm_deviation": abs(norm64 - 1), "max_abs_diff": maxdiff}
    plain.close()
    return out


def batch_leg(count, seed=20250404, direct=False, tuning=None, precisions=(1, 3)):
    """512 variational circuits (12-22 qubits, 4-16 layers of RY/RZ + CNOT ladder): one
    autotuned hipGraph launch (complex64 states, FP64 <Z> reductions) against the per-circuit
    plain-method loop in C++ (complex128, one kernel per gate, one simulator per qubit
    count; qcs_ext_batch_run_plain).  The block products of the circuits in HBM run on FP32
    MFMA (the top-level figures) and on BF16x3 split-precision MFMA ("bf16x3"), each with its
    own tuning and its own accuracy against the plain loop."""
    lib = pyqcs.gpu_library()
    work = circuits.variational_batch(count, seed=seed)
    gates = sum(len(g) for _, g in work)
    b = pyqcs.Batch(lib)
    for n, g in work:
        b.add(n, g)
    z_plain, t_plain = b.run_plain()
    b.close()
    log(f"batch leg: {count} circuits, {gates} gates; plain loop {t_plain:.3f}s")
    legs = {}
    for mode in precisions:
        b = pyqcs.Batch(lib)
        for n, g in work:
            b.add(n, g)
        b.set_precision(mode)
        t0 = time.perf_counter()
        # the autotuner times graph replays; a direct-launch (profiler) run takes the tuning
        # given on the command line, or the defaults
        if tuning is not None:
            b.set_tuning(*tuning)
            tun = dict(zip(("lds_max_qubits", "block_size", "block_qubits", "streams", "stage_bits"), tuning))
        elif direct:
            tun = {"default": True}
        else:
            tun = b.autotune()
        t_tune = time.perf_counter() - t0
        b.run()
        runs = []
        for _ in range(5):
            t0 = time.perf_counter()
            z_batch, dev = b.run_direct() if direct else b.run()
            runs.append((time.perf_counter() - t0, dev))
        info = b.info()
        traffic = b.traffic()
        b.close()
        wall = min(r[0] for r in runs)
        dev = min(r[1] for r in runs)
        gbps = traffic["hbm_bytes"] / dev / 1e9
        err = max(float(abs(x - y).max()) for x, y in zip(z_batch, z_plain))
        name = {1: "FP32", 3: "BF16x3"}[mode]
        log(f"batch leg ({name} MFMA): graph {dev * 1e3:.2f} ms device ({wall * 1e3:.2f} ms wall), "
            f"{t_plain / wall:.1f}x the plain loop, max |d<Z>| {err:.2e}; tuning {tun} found in {t_tune:.1f}s")
        log(f"batch leg ({name} MFMA): {traffic['hbm_bytes'] / 1e9:.1f} GB algorithmic HBM traffic in "
            f"{traffic['kernel_launches']} launches: {gbps:.0f} GB/s over the whole run")
        legs[mode] = {"mfma": name, "graph_device_s": dev, "graph_wall_s": wall,
                      "speedup_wall": t_plain / wall, "gates_per_s": gates / wall,
                      "max_abs_diff_expz": err, "tuning": tun, "autotune_s": t_tune,
                      "graph_nodes": info["graph_nodes"], "hbm_bytes": traffic["hbm_bytes"],
                      "kernel_launches": traffic["kernel_launches"], "hbm_GBps_whole_run": gbps,
                      "hbm_frac_whole_run": gbps / 8000.0}
    first = legs[precisions[0]]
    out = {"config": f"{count} variational circuits, 12-22 qubits, 4-16 layers RY+RZ on every "
                     f"qubit + CNOT ladder, {gates} gates; <Z_i> of every qubit",
           "circuits": count, "gates": gates, "plain_loop_s": t_plain,
           "launch": "direct" if direct else "graph"}
    out.update(first)
    if 3 in legs and precisions[0] != 3:
        out["bf16x3"] = legs[3]
    return out


def _class_rate(sim, cls):
    """Launches, average ms and algorithmic GB/s of one kernel class since the last reset."""
    v = sim.profile_get().get(cls)
    if not v:
        return None
    avg = v["seconds"] / v["launches"]
    gbs = v["bytes"] / v["seconds"] / 1e9
    return {"launches": v["launches"], "avg_ms": avg * 1e3, "GBps": gbs, "frac": gbs / (HBM_PEAK / 1e9)}


SUBSYSTEM_GATES = (
    # (gate, parameter count, kernel class, operand tuples as functions of n)
    ("rz", 1, "diag", lambda n: [(0,), (5,), (17,), (n - 1,)]),
    ("rzz", 1, "diag", lambda n: [(0, 1), (14, 15), (n - 2, n - 1)]),
    ("rxx", 1, "dense4", lambda n: [(0, 1), (3, 4), (14, 15), (n - 3, n - 1)]),
    ("ecr", 0, "dense4", lambda n: [(0, 1), (14, 15), (n - 2, n - 1)]),
    ("dcx", 0, "mono", lambda n: [(0, 1), (14, 15), (n - 2, n - 1)]),
    ("rccx", 0, "mono", lambda n: [(0, 1, 2), (14, 15, 16), (n - 3, n - 2, n - 1)]),
    ("swap", 0, "pair", lambda n: [(0, 1), (1, 2), (0, n - 1), (14, 15), (n - 2, n - 1)]),
    ("u3", 3, "pair", lambda n: [(t,) for t in range(n)]),
    # (targets, controls): a control on qubit 0 (the GHZ chain's CX), and the MCX of the
    # headline circuit with its controls high and low
    ("x", 0, "pair", lambda n: [((n - 1,), (0,)), ((5,), (0,)), ((n - 1,), (n - 4, n - 3, n - 2)), ((n - 1,), (0, 1, 2))]),
)


def subsystem_leg(n=30, reps=4):
    """Every kernel family of the plain method on an n-qubit complex128 state (one random
    brick layer, so every amplitude is non-zero), timed with HIP events around each launch:
    algorithmic bytes per launch (2 * 16 B * amplitudes the gate may change; a permutation
    pass one sweep; a measurement's {p0,p1} reduction one read of the state, its collapse
    the zeroed half, plus a read and write of the kept half when renormalising; the
    sampling prefix one read) over the average launch time, against 8 TB/s.  Per gate and
    operand position, since low operands (qubits 0..2, 16-48 B apart) are the hard case.
    The measurement cases also give the reference's per-qubit sampling path (measure every
    qubit in turn, src/qcs_main.cpp:153-193, src/qcs.cu:2545-2677) as wall time."""
    lib = pyqcs.gpu_library()
    sim = pyqcs.Simulator(lib, n, seed=7)
    prep = circuits.brick(n, 1, seed=CIRCUIT_SEED + 21)

    def fresh():
        sim.profile(False)
        sim.call("set_zero_state")
        sim.run(prep)
        sim.flush()
        sim.norm()

    out = {"config": f"{n} qubits complex128, state of one random brick layer; {reps} launches per case"}
    fresh()
    gates = {}
    for name, npar, cls, ops in SUBSYSTEM_GATES:
        rows = []
        for opnd in ops(n):
            tg, ctl = opnd if isinstance(opnd[0], tuple) else (opnd, ())
            params = tuple(0.3 + 0.1 * i for i in range(npar))
            sim.profile_reset()
            sim.profile(True)
            for _ in range(reps):
                sim.gate(name, tg, params, ctrls=ctl)
            r = _class_rate(sim, cls)
            sim.profile(False)
            del r["launches"]  # reps
            r["operands"] = list(tg)
            if ctl:
                r["controls"] = list(ctl)
            rows.append(r)
            log(f"subsystems: {name}{tuple(tg)}{' ctrl ' + str(tuple(ctl)) if ctl else ''} {cls}: "
                f"{r['avg_ms']:.3f} ms, {r['GBps']:.0f} GB/s ({r['frac']:.2f})")
        gates[name if name != "x" else "controlled_x"] = rows
    out["gates"] = gates
    ident = list(range(n))
    rng = np.random.default_rng(CIRCUIT_SEED)
    low_high = ident.copy()
    for a, b in ((0, n - 3), (1, n - 1), (2, n - 5), (9, 14)):
        low_high[a], low_high[b] = low_high[b], low_high[a]
    cases = {"low_high_4_pairs": low_high, "reversal": ident[::-1],
             "random": [int(q) for q in rng.permutation(n)]}
    perm = {}
    for name, want in cases.items():
        sim.profile_reset()
        sim.profile(True)
        t0 = time.perf_counter()
        sim.permute(want)
        sim.flush()
        sim.norm()
        dt = time.perf_counter() - t0
        r = _class_rate(sim, "permute")
        sim.profile(False)
        sim.permute(ident)
        r["passes"] = r["launches"]
        perm[name] = r
        log(f"subsystems: permute {name}: {r['launches']} passes, {r['avg_ms']:.3f} ms per pass, "
            f"{r['GBps']:.0f} GB/s ({r['frac']:.2f})")
    out["permute"] = perm
    meas = {}
    for renorm in (False, True):
        sim.set_renormalize(renorm)
        key = "renormalised" if renorm else "plain"
        rows = []
        for q in (0, n // 2, n - 1):
            fresh()
            sim.profile_reset()
            sim.profile(True)
            sim.measure(q)
            red, col = _class_rate(sim, "reduce"), _class_rate(sim, "collapse")
            sim.profile(False)
            rows.append({"qubit": q, "reduce": red, "collapse": col})
            log(f"subsystems: measure q{q} ({key}): reduce {red['avg_ms']:.3f} ms {red['GBps']:.0f} GB/s, "
                f"collapse {col['avg_ms']:.3f} ms {col['GBps']:.0f} GB/s")
        fresh()
        t0 = time.perf_counter()
        bits = [sim.measure(q) for q in range(n)]
        dt = time.perf_counter() - t0
        meas[key] = {"first_measure_by_qubit": rows, "all_qubits_s": dt, "outcome": "".join(map(str, bits))}
        log(f"subsystems: measure all {n} qubits in turn ({key}): {dt * 1e3:.1f} ms")
    sim.set_renormalize(False)
    out["measure"] = meas
    fresh()
    sim.profile_reset()
    sim.profile(True)
    sim.probability_total()
    fold = _class_rate(sim, "reduce")
    sim.sample(4096, seed=SAMPLE_SEED)
    sim.profile(False)
    out["prefix_fold"] = fold
    log(f"subsystems: sampling prefix {fold['avg_ms']:.3f} ms, {fold['GBps']:.0f} GB/s ({fold['frac']:.2f})")
    sim.close()
    return out


def _timed_run(sim, circ, prep=(), reps=1, runs=None):
    """Median seconds of: gates queued and applied (flush) plus a norm; the state is reset
    to |0...0> and `prep` applied (untimed) before each repetition.  Every repetition's
    seconds are appended to `runs` when given."""
    ts = runs if runs is not None else []
    for _ in range(reps):
        sim.call("set_zero_state")
        if prep:
            sim.run(prep)
        sim.flush()
        sim.norm()
        t0 = time.perf_counter()
        sim.run(circ)
        sim.flush()
        sim.norm()
        ts.append(time.perf_counter() - t0)
    return float(np.median(ts))


def planner_leg(n, depth, record_count, k=4, fixed_sweep=False):
    """Learned fusion planner on complex128 fused blocks (the workloads of the planner
    configuration): a cost model trained on the GPU on recorded launch timings (random
    blocks and stages at 26-32 qubits, and every candidate stage plan's launches on
    training circuits at 26-30 qubits, none of them the evaluated circuits), then an n-qubit
    QFT on the state of one random brick layer and an n-qubit brick circuit of the given
    depth, each run four ways -- the greedy fusion fallback (one sweep per block), the
    stage plan that a model is compared with, circuit passes (the default without a model), and
    the plan the model picks (taken only when its predicted gain
    over the default exceeds the model's error; one run each, so an override runs as the
    model picked it, before the planner's measured check has compared it with the default)
    -- and each output compared with a second state in HBM, whose gates are called one by
    one: a kernel per gate, which shares no code with passes or stages."""
    lib = pyqcs.gpu_library()
    model, info = pyqcs.train_cost_model(lib, 2, k, (26, 28, 30, 32), record_count, (26, 28, 30), log=log)
    out = {"config": f"complex128 fused blocks (k<={k}), {n}-qubit QFT on a random brick layer and "
                     f"{n}-qubit brick depth {depth}; outputs against complex128 gate by gate",
           "cost_model": info}
    prep_qft = circuits.brick(n, 1, seed=CIRCUIT_SEED + 9)
    work = {"qft": (prep_qft, circuits.qft(n)), "brick": ((), circuits.brick(n, depth, seed=CIRCUIT_SEED + 5))}
    try:
        fused = pyqcs.Simulator(lib, n, seed=1, precision=2, block_qubits=k)
        plain = pyqcs.Simulator(lib, n, seed=1)
    except pyqcs.QcsError:
        n -= 1  # two complex128 states must fit in HBM
        log(f"planner leg: two {n + 1}-qubit states do not fit; {n} qubits")
        out["qubits_fallback"] = n
        prep_qft = circuits.brick(n, 1, seed=CIRCUIT_SEED + 9)
        work = {"qft": (prep_qft, circuits.qft(n)), "brick": ((), circuits.brick(n, depth, seed=CIRCUIT_SEED + 5))}
        fused = pyqcs.Simulator(lib, n, seed=1, precision=2, block_qubits=k)
        plain = pyqcs.Simulator(lib, n, seed=1)
    out["qubits"] = n
    try:
        for name, (prep, circ) in work.items():
            res = {"gates": len(circ)}
            plain.call("set_zero_state")
            for op in prep:
                plain.gate(*op)
            plain.norm()
            t0 = time.perf_counter()
            for op in circ:
                plain.gate(*op)
            plain.norm()
            res["plain_per_gate_s"] = time.perf_counter() - t0
            for mode in ("greedy", "stages", "passes", "learned"):
                pyqcs.set_planner(fused, model if mode == "learned" else None)
                if mode == "greedy":
                    fused.set_plan(0, k, window=64, rule=0)
                elif mode == "stages":
                    fused.set_plan(12, min(k, 3), tiles=2)
                else:
                    fused.set_plan(None)
                _, b0 = fused.fusion_stats()
                st0 = pyqcs.planner_stats(fused)
                dt = _timed_run(fused, circ, prep)
                _, b1 = fused.fusion_stats()
                ov, maxdiff = fused.overlap(plain)
                fid = abs(ov) ** 2 / (fused.norm() * plain.norm())
                res[f"{mode}_s"] = dt
                res[f"{mode}_sweeps"] = b1 - b0
                res[f"{mode}_fidelity_vs_per_gate"] = fid
                res[f"{mode}_max_abs_diff_vs_per_gate"] = maxdiff
                if mode == "learned":
                    st1 = pyqcs.planner_stats(fused)
                    res["learned_choices"] = st1["learned_choices"] - st0["learned_choices"]
                    res["flushes"] = st1["flushes"] - st0["flushes"]
                    res["learned_plan"] = list(pyqcs.planner_last_choice(fused))
                log(f"planner leg: {name} {mode}: {dt:.3f}s, {b1 - b0} sweeps, fidelity vs per-gate "
                    f"{fid:.15f}, max|d| {maxdiff:.2e}")
            pyqcs.set_planner(fused, None)
            if fixed_sweep:
                fixed = {}
                for m in (11, 12, 13):
                    for kb in (3, 4):
                        for tiles in (0, 1):
                            fused.set_plan(m, kb, tiles=tiles)
                            fixed[f"{m}/{kb}/{'window' if tiles else 'grow'}"] = _timed_run(fused, circ, prep)
                res["fixed_plans_s"] = fixed
                best = min(fixed, key=fixed.get)
                log(f"planner leg: {name}: best fixed stage plan {best} {fixed[best]:.3f}s; "
                    + " ".join(f"{p}={t:.3f}" for p, t in fixed.items()))
            fused.set_plan(None)
            res["learned_vs_stages"] = res["stages_s"] / res["learned_s"]
            res["learned_vs_greedy"] = res["greedy_s"] / res["learned_s"]
            res["stages_vs_greedy"] = res["greedy_s"] / res["stages_s"]
            log(f"planner leg: {name}: learned vs default stages {res['learned_vs_stages']:.3f}x, "
                f"vs greedy {res['learned_vs_greedy']:.2f}x; per gate {res['plain_per_gate_s']:.2f}s")
            out[name] = res
    finally:
        pyqcs.set_planner(fused, None)
        fused.close()
        plain.close()
        model.close()
    return out


PRECISION_PLANNER_WORKLOADS = ("qft", "brick", "qaoa", "narrow", "random2q", "diagonal")


def precision_planner_workloads(n):
    """Evaluation circuits of the precision-form planner leg (seeds outside the training
    set): prep and circuit per workload."""
    return {"qft": (circuits.brick(n, 1, seed=CIRCUIT_SEED + 9), circuits.qft(n)),
            "brick": ((), circuits.brick(n, 32, seed=CIRCUIT_SEED + 3)),
            "qaoa": ((), circuits.qaoa_ring(n, 3, CIRCUIT_SEED + 11)),
            "narrow": ((), circuits.narrow_random(n, 10, 300, CIRCUIT_SEED + 12)),
            "random2q": ((), circuits.random_two_qubit(n, 400, CIRCUIT_SEED + 13)),
            "diagonal": ((), circuits.diagonal_heavy(n, 400, CIRCUIT_SEED + 14))}


def precision_planner_leg(n, record_count, fixed_sweep=False):
    """The learned planner in the precision form (complex64 state, BF16x3 stages of 4- or
    5-qubit blocks on 2^11-2^14-amplitude tiles): cost model trained as in the complex128
    leg, then six n-qubit workloads run with the default stage plan (2^13 tiles, 5-qubit
    blocks, fewer-stage tile choice) and with the model's choice (median of 3 runs each).
    With fixed_sweep, every fixed stage plan is timed as well."""
    lib = pyqcs.gpu_library()
    # With the planner's measured check (on by default), a circuit's first run takes the
    # model's choice, its second the default plan, and the third the faster of the two
    # (when the model keeps the default, all three run it): learned_s is the median.
    # candidate-plan timings at 30 and 32 qubits (one seed): the launches of the sizes the
    # model chooses for, at the recording cost of three seeds at 26-30 qubits
    model, info = pyqcs.train_cost_model(lib, 3, 5, (26, 28, 30, 32), record_count // 2, (30, 32), plan_seeds=(1001,), log=log)
    out = {"config": f"complex64 BF16x3 stages, {n} qubits; workloads {', '.join(PRECISION_PLANNER_WORKLOADS)}",
           "cost_model": info}
    sim = pyqcs.Simulator(lib, n, seed=1, precision=3, block_qubits=5)
    try:
        for name, (prep, circ) in precision_planner_workloads(n).items():
            res = {"gates": len(circ)}
            pyqcs.set_planner(sim, None)
            res["default_s"] = _timed_run(sim, circ, prep, reps=3)
            pyqcs.set_planner(sim, model)
            st0 = pyqcs.planner_stats(sim)
            runs = []
            res["learned_s"] = _timed_run(sim, circ, prep, reps=3, runs=runs)
            st1 = pyqcs.planner_stats(sim)
            res["learned_runs_s"] = runs
            res["learned_plan"] = list(pyqcs.planner_last_choice(sim))
            # flushes that ran the model's (non-default) choice over the 3 runs and preps
            res["learned_flushes"] = st1["learned_choices"] - st0["learned_choices"]
            res["flushes"] = st1["flushes"] - st0["flushes"]
            pyqcs.set_planner(sim, None)
            res["learned_vs_default"] = res["default_s"] / res["learned_s"]
            if fixed_sweep:
                fixed = {}
                for m in (11, 12, 13, 14):
                    for kb in (4, 5):
                        for tiles in (0, 1):
                            sim.set_plan(m, kb, tiles=tiles)
                            fixed[f"{m}/{kb}/{'window' if tiles else 'grow'}"] = _timed_run(sim, circ, prep, reps=3)
                sim.set_plan(None)
                res["fixed_plans_s"] = fixed
            log(f"precision planner leg: {name}: default {res['default_s'] * 1e3:.1f} ms, learned "
                f"{res['learned_s'] * 1e3:.1f} ms ({res['learned_vs_default']:.3f}x; runs "
                + ", ".join(f"{t * 1e3:.1f}" for t in runs)
                + f"; {res['learned_flushes']:.0f} of {res['flushes']:.0f} flushes off the default plan), plan {res['learned_plan']}")
            out[name] = res
        if fixed_sweep:
            # the best single fixed plan over all workloads, against the learned choices
            names = list(out[PRECISION_PLANNER_WORKLOADS[0]]["fixed_plans_s"])
            totals = {p: sum(out[w]["fixed_plans_s"][p] for w in PRECISION_PLANNER_WORKLOADS) for p in names}
            best = min(totals, key=totals.get)
            out["best_fixed_plan"] = best
            out["best_fixed_total_s"] = totals[best]
        out["default_total_s"] = sum(out[w]["default_s"] for w in PRECISION_PLANNER_WORKLOADS)
        out["learned_total_s"] = sum(out[w]["learned_s"] for w in PRECISION_PLANNER_WORKLOADS)
        log(f"precision planner leg: total default {out['default_total_s']:.3f}s, learned {out['learned_total_s']:.3f}s"
            + (f", best fixed plan {out['best_fixed_plan']} {out['best_fixed_total_s']:.3f}s" if fixed_sweep else ""))
    finally:
        pyqcs.set_planner(sim, None)
        sim.close()
        model.close()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--qubits", type=int, default=30)
    ap.add_argument("--depth", type=int, default=24)
    ap.add_argument("--shots", type=int, default=4096)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-budget", type=float, default=20.0)
    ap.add_argument("--no-fused", action="store_true")
    ap.add_argument("--fused-qubits", type=int, default=32)
    ap.add_argument("--fused-depth", type=int, default=32)
    ap.add_argument("--fused-k", type=int, default=5)
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--batch-circuits", type=int, default=512)
    ap.add_argument("--batch-tuning", type=lambda s: tuple(int(v) for v in s.split(",")), default=None,
                    help="lds_max_qubits,block_size,block_qubits,streams,stage_bits instead of the autotuner")
    ap.add_argument("--batch-no-graph", action="store_true",
                    help="issue the batch's launches directly instead of one graph launch "
                         "(same kernels; for profilers that do not follow graph launches)")
    ap.add_argument("--no-planner", action="store_true")
    ap.add_argument("--no-subsystems", action="store_true",
                    help="skip the per-kernel-family leg (diagonal, 4x4, monomial, swap, "
                         "permutation, measurement, prefix) at the headline size")
    ap.add_argument("--no-small", action="store_true", help="skip the 20-qubit GPU-vs-CPU leg")
    ap.add_argument("--planner-qubits", type=int, default=33)
    ap.add_argument("--planner-depth", type=int, default=40)
    ap.add_argument("--planner-k", type=int, default=4)
    ap.add_argument("--planner-record", type=int, default=10000,
                    help="random blocks and stages timed for the complex128 cost model over 26, 28, "
                         "30 and 32 qubits (8:4:2:1; half as many for the precision-form model), "
                         "besides the launches of the candidate plans of the training circuits")
    ap.add_argument("--planner-fixed-sweep", action="store_true",
                    help="also time every fixed stage plan on the planner workloads (both legs)")
    ap.add_argument("--calibrate", action="store_true",
                    help="also run one write-only fill and one read-only norm pass of the "
                         "full state (known HBM bytes, for scaling PMC byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for {args.gpus}); the multi-GPU "
              "sharding is a design, not part of this build", file=sys.stderr)
        sys.exit(2)

    n = args.qubits
    circ = circuits.brick(n, args.depth, seed=CIRCUIT_SEED, mcx=4)
    ngates = len(circ)
    alg_bytes = sum(circuits.algorithmic_bytes(n, op) for op in circ)
    log(f"workload: {n} qubits, depth {args.depth}, {ngates} gates, {alg_bytes / 1e12:.2f} TB algorithmic")

    lib = pyqcs.gpu_library()
    sim = pyqcs.Simulator(lib, n, seed=1)

    def step():
        sim.call("set_zero_state")
        sim.run(circ)
        total = sim.probability_total()
        out = sim.sample(args.shots, seed=SAMPLE_SEED)
        return total, out

    for i in range(args.warmup):
        t0 = time.perf_counter()
        total, _ = step()
        log(f"warmup {i}: {time.perf_counter() - t0:.3f}s total prob {total:.15f}")

    sim.profile_reset()
    sim.profile(True)
    e0, e1 = sim.event_create(), sim.event_create()
    sim.flush()
    t0 = time.perf_counter()
    sim.event_record(e0)
    for i in range(args.steps):
        ts = time.perf_counter()
        total, out = step()
        log(f"step {i}: {time.perf_counter() - ts:.3f}s")
    sim.event_record(e1)
    gpu_s = sim.elapsed(e0, e1)
    wall = time.perf_counter() - t0
    prof = sim.profile_get()
    sim.profile(False)
    log(f"timed: wall {wall:.3f}s, stream events {gpu_s:.3f}s")
    for k, v in prof.items():
        gbs = v["bytes"] / v["seconds"] / 1e9 if v["seconds"] else 0
        log(f"  {k:9s} launches {v['launches']:6d}  {v['seconds']:.4f}s  avg {v['seconds'] / v['launches'] * 1e3:.3f} ms  {gbs:.1f} GB/s")
    if args.calibrate:
        sim.call("set_zero_state")  # writes 16 * 2^n bytes
        log(f"calibration norm {sim.norm():.3f}")  # reads 16 * 2^n bytes
    sim.close()

    passes = prof.get("fused", {"launches": 1, "seconds": 1, "bytes": 0})
    achieved = passes["bytes"] / passes["seconds"] / 1e9
    traffic = traffic_from_profiles()

    result = {
        "metric": "gates/s + % HBM roofline, 30q complex128; fused c64 speedup at fidelity>=1-1e-6",
        "value": ngates * args.steps / wall,
        "unit": "gates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": wall / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded SplitMix64 circuit parameters and sampling uniforms)",
        "config": {
            "workload": f"brick{n}_c128: {n} qubits complex128, {args.depth} brick layers "
                        f"(U3 all + CZ even/odd), 4 MCX with 3 controls, full probability "
                        f"reduction + {args.shots} samples",
            "qubits": n, "depth": args.depth, "gates": ngates, "shots": args.shots,
            "circuit_seed": CIRCUIT_SEED, "sample_seed": SAMPLE_SEED,
            "method": "plain: whole circuit per call, one kernel per sweep of the state",
            "sweeps_per_step": passes["launches"] / args.steps,
        },
        "roofline": {
            "bound": "hbm",
            "kernel": "k_pass (HIP events over the timed steps)",
            "achieved": achieved,
            "peak": HBM_PEAK / 1e9,
            "unit": "GB/s",
            "frac": achieved / (HBM_PEAK / 1e9),
            "traffic": traffic,
        },
        # what one sweep per gate would move, over the time taken; and what was moved
        "sweeps_per_s": alg_bytes / (2 * 16 * (1 << n)) * args.steps / wall,
        "hbm_frac_whole_step": sum(v["bytes"] for v in prof.values()) / wall / HBM_PEAK,
    }
    if not args.no_subsystems:
        result["subsystems"] = subsystem_leg(n)
    if not args.no_small:
        result["small_20q"] = small_leg()
    if not args.no_fused:
        result["fused_qft"] = qft_c64_leg(args.fused_qubits)
    if not args.no_fused:
        result.update(fused_leg(args.fused_qubits, args.fused_depth, args.fused_k, args.shots))
    if not args.no_batch:
        result["batch"] = batch_leg(args.batch_circuits, direct=args.batch_no_graph, tuning=args.batch_tuning)
    if not args.no_planner:
        result["planner"] = planner_leg(args.planner_qubits, args.planner_depth, args.planner_record, args.planner_k,
                                        fixed_sweep=args.planner_fixed_sweep)
        result["planner_precision"] = precision_planner_leg(args.fused_qubits, args.planner_record,
                                                            fixed_sweep=args.planner_fixed_sweep)
    if not args.no_cpu_baseline:
        result["cpu_baseline"] = cpu_baseline(n, circ, args.cpu_budget)
    line = json.dumps({**brief(result), "value": result["value"], "ms_per_step": result["ms_per_step"]}, separators=(",", ":"))
    log(f"result line: {len(line)} characters")
    print(line, flush=True)


if __name__ == "__main__":
    main()
