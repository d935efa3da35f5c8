"""The gates that the device hands to its backend at once: bounded in number
and in the bytes of their matrices, in order, none lost (no GPU)."""
import numpy as np
import pytest
from test_device_cpu import FakeBackend, FakeSV

from pennylane_lightning_gpu import circuit as qc
from pennylane_lightning_gpu import lightning_gpu as lg


class SequenceSV(FakeSV):
    def applySequence(self, names, wires, inverses, params, matrices):
        self.calls.append(("applySequence", names, wires, inverses, params, matrices))


class SequenceBackend(FakeBackend):
    LightningGPU_C128 = SequenceSV
    LightningGPU_C64 = SequenceSV


def matrix_op(k):
    return qc.Operation("QubitUnitary", list(range(k)), [], matrix=np.eye(1 << k))


@pytest.mark.parametrize("ks", [[8] * 40, [10, 1, 10, 10, 2], [2] * 300, []])
def test_matrices_held_at_once_are_bounded(ks):
    dev = lg.LightningGPU(12, _backend=SequenceBackend)
    ops = []
    for i, k in enumerate(ks):
        ops += [qc.Operation("RX", [i % 12], [0.1 * i]), matrix_op(k)]
    ops.append(qc.Operation("PauliX", [0]))
    dev.apply_cq(ops)
    seqs = [c for c in dev._gpu_state.calls if c[0] == "applySequence"]
    largest = max([16 << 2 * k for k in ks] + [0])
    for _, names, wires, inverses, params, mats in seqs:
        assert len(names) == len(wires) == len(inverses) == len(params) == len(mats) <= lg._SEQUENCE_MAX
        assert sum(m.nbytes for m in mats) < lg._SEQUENCE_MATRIX_BYTES + largest
    assert [n for c in seqs for n in c[1]] == [o.name for o in ops]
    assert [p for c in seqs for p in c[4]] == [[float(x) for x in o.parameters] if o.name == "RX" else [] for o in ops]


def test_gates_before_a_refused_one_are_applied():
    dev = lg.LightningGPU(3, _backend=SequenceBackend)
    bad = qc.Operation("QubitUnitary", [0], [], matrix=np.zeros((0, 0)))
    with pytest.raises(Exception):
        dev.apply_cq([qc.Operation("PauliX", [0]), qc.Operation("RY", [1], [0.5]), bad, qc.Operation("PauliZ", [2])])
    seqs = [c for c in dev._gpu_state.calls if c[0] == "applySequence"]
    assert [n for c in seqs for n in c[1]] == ["PauliX", "RY"]
