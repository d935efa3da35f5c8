"""The device applies a circuit's gates together where the backend state takes
a sequence (complex128): the same state as one gate at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("pennylane_lightning_gpu._native")

from pennylane_lightning_gpu import circuit as qc  # noqa: E402
from pennylane_lightning_gpu.lightning_gpu import _SEQUENCE_MAX, LightningGPU  # noqa: E402


def random_ops(n, count, seed):
    rng = np.random.default_rng(seed)
    ops = []
    for _ in range(count):
        w = [int(x) for x in rng.permutation(n)[:3]]
        k = int(rng.integers(8))
        if k < 3:
            ops.append(qc.Operation(("RX", "RY", "RZ")[k], w[:1], [float(rng.normal())]))
        elif k == 3:
            ops.append(qc.Operation("CNOT", w[:2]))
        elif k == 4:
            ops.append(qc.Adjoint(qc.Operation("CRY", w[:2], [float(rng.normal())])))
        elif k == 5:
            ops.append(qc.Operation("Rot", w[:1], list(rng.normal(size=3))))
        elif k == 6:
            u, _ = np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))
            op = qc.Operation("QubitUnitary", w[:2], [], matrix=u)
            ops.append(qc.Adjoint(op) if rng.integers(2) else op)
        else:
            ops.append(qc.Operation("Identity", w[:1]))
    return ops


@pytest.mark.parametrize("n,count", [(4, 1), (4, 30), (11, 200), (14, _SEQUENCE_MAX + 300)])
def test_sequence_equals_gates_one_by_one(n, count):
    ops = random_ops(n, count, n + count)
    dev, one = LightningGPU(n), LightningGPU(n)
    dev.apply(ops)
    for o in ops:
        one.apply_cq([o])
    # each gate rounds an amplitude a few times: error below 8 eps per gate
    np.testing.assert_allclose(dev.state, one.state, atol=8 * 2.3e-16 * max(8, count), rtol=0)


def test_complex64_applies_gates_one_by_one():
    assert not hasattr(LightningGPU(3, c_dtype=np.complex64)._gpu_state, "applySequence")
