"""The tests that were written for the kernels of single gates, of blocks and of stages, once more
with those kernels chosen: Simulator.run on complex128 states and the default flush of modes 1
and 2 run circuit passes, which those kernels serve beside (single calls, measured qubits, a
window of local qubits, fixed plans, gates that passes do not take).

Complex128 states go gate by gate here (run() calls a subclass's own gate()), and the classes of
the launches that the profile counts must be the ones the test is for, and no sweep of several
gates; the fused modes are asked for stages, which turns passes off."""
import collections

import pytest

import pyqcs
import test_gpu_fused as fused
import test_gpu_parity as parity

pytestmark = pytest.mark.gpu

Plain = pyqcs.Simulator


class GateByGate(Plain):
    seen = collections.Counter()

    def __init__(self, library, *args, **kw):
        super().__init__(library, *args, **kw)
        self.counted = library.path == pyqcs.GPU_LIB and not kw.get("precision")
        if self.counted:
            self.profile(True)

    def gate(self, *args, **kw):
        super().gate(*args, **kw)

    def close(self):
        if getattr(self, "counted", False) and self.h is not None:
            for name, v in self.profile_get().items():
                GateByGate.seen[name] += v["launches"]
        super().close()


class Stages(Plain):
    def __init__(self, library, *args, **kw):
        super().__init__(library, *args, **kw)
        if kw.get("precision") in (1, 2) and kw.get("stage_bits") is None:
            self.set_stage_bits(13)  # the tile bits that are the default


GATES = {"pair", "phase", "diag", "dense4", "mono"}


@pytest.mark.parametrize("test,args,classes", [
    (parity.test_low_target_pair_kernel, (), {"pair"}),
    (parity.test_low_operand_phase_kernel, (), {"phase"}),
    (parity.test_low_operand_gate_kernel, (), GATES),
    (parity.test_random_circuit_all_gates, (), GATES),
    (parity.test_cached_size_all_gates, (22,), GATES),
    (parity.test_cached_size_all_gates, (24,), GATES),
    (parity.test_config_ghz_u3_cz_20q, (), {"pair", "phase"}),
    (parity.test_measurement_sequences, (), {"pair"}),
    (parity.test_renormalize, (), {"pair", "phase"}),
    (parity.test_local_window_and_permute, (), {"pair"}),
], ids=lambda v: getattr(v, "__name__", None))
def test_kernels_of_single_gates(gpu, oracle, monkeypatch, test, args, classes):
    monkeypatch.setattr(pyqcs, "Simulator", GateByGate)
    GateByGate.seen.clear()
    test(gpu, oracle, *args)
    print(dict(GateByGate.seen), flush=True)
    assert GateByGate.seen["fused"] == 0
    assert all(GateByGate.seen[c] > 0 for c in classes)


# complex64 states against complex128 ones whose gates run one by one: not the same code twice
@pytest.mark.parametrize("test,args", [(fused.test_overlap_with_plain_gpu_path, (1,)), (fused.test_overlap_with_plain_gpu_path, (3,)),
                                       (fused.test_unnormalised_overlap_22q, (1, "brick")), (fused.test_unnormalised_overlap_22q, (3, "qft"))])
def test_references_gate_by_gate(gpu, monkeypatch, test, args):
    monkeypatch.setattr(pyqcs, "Simulator", GateByGate)
    GateByGate.seen.clear()
    test(gpu, *args)
    assert GateByGate.seen["fused"] == 0 and GateByGate.seen["pair"] > 0


@pytest.mark.parametrize("test,args", [
    (fused.test_random_all_gates, (4, 1)), (fused.test_random_all_gates, (5, 1)),
    (fused.test_each_gate_single, (1,)), (fused.test_wide_gates, ()), (fused.test_brick_mapping_and_fusion_counts, (1,)),
    (fused.test_measure_sample_in_fused_mode, ()), (fused.test_window_in_fused_mode, ()),
    (fused.test_fused_complex128_matches_oracle, ()), (fused.test_fused_complex128_qft_and_measure, ()),
    (fused.test_stages_complex128_match_oracle, (3,)), (fused.test_stages_complex128_match_oracle, (4,)),
    (fused.test_stages_complex128_diagonal, (3,)), (fused.test_stages_complex128_diagonal, (4,)),
], ids=lambda v: getattr(v, "__name__", None))
def test_kernels_of_blocks_and_stages(gpu, oracle, monkeypatch, test, args):
    monkeypatch.setattr(pyqcs, "Simulator", Stages)
    test(gpu, oracle, *args)
