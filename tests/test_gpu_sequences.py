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


N = pytest.importorskip("pennylane_lightning_gpu._native")


def rand_state(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return v / np.linalg.norm(v)


@pytest.mark.parametrize("n", [3, 10, 12, 13, 15])
def test_sum_of_pauli_words(n):
    """dst = sum c P src against one word at a time: several passes, words wider than a tile, many words of one flip
    mask, every number of Y factors, identities, no word at all; dst's old contents do not matter."""
    rng = np.random.default_rng(n)
    words, wires = ["X" * n, "Y" * n, "Z" * n, "", "II"], [list(range(n))] * 3 + [[], [0, n - 1]]
    for k in range(60):
        ws = [int(x) for x in rng.permutation(n)[:int(rng.integers(1, min(n, 5) + 1))]]
        words.append("".join(rng.choice(list("XYZ"), len(ws))) if k % 2 else "Z" * len(ws))
        wires.append(ws)
    coeffs = rng.normal(size=len(words))
    for dtype, tol in ((np.complex128, 1e-14), (np.complex64, 1e-5)):
        src = N.State(n, dtype).upload(rand_state(n, n).astype(dtype))
        dst = N.State(n, dtype).upload(rand_state(n, n + 1).astype(dtype))
        for use in (list(range(len(words))), [1], [2, 7], []):
            chars = "".join(words[w] for w in use).encode()
            wf = np.array([x for w in use for x in wires[w]] or [0], dtype=np.int32)
            offs = np.concatenate([[0], np.cumsum([len(words[w]) for w in use])]).astype(np.int64)
            c = np.array([coeffs[w] for w in use] or [0.0])
            fn = N.lib().lgh_sv_pauli_sum_from
            fn.argtypes = [N.C.c_void_p, N.C.c_void_p, N.C.c_int64, N.C.c_char_p] + [N.C.c_void_p] * 3
            N.check(fn(dst.handle, src.handle, len(use), chars, wf.ctypes.data, offs.ctypes.data, c.ctypes.data))
            ref, one = np.zeros(1 << n, dtype=np.complex128), N.State(n, dtype)
            for w in use:
                ref += coeffs[w] * one.set_pauli_word_of(src, words[w], wires[w]).download()
            # |amplitude| < 1, 65 terms of size ~1: error below 65 eps, and a rounding in the state's precision
            np.testing.assert_allclose(dst.download(), ref, atol=tol, rtol=0)


@pytest.mark.parametrize("n", [6, 11, 15])
def test_gates_on_pairs_of_basis_states(n):
    """Excitations, swaps and IsingXX / YY, forward and in the adjoint sweep, between and at the ends of fused passes,
    trainable or not, against the oracle; the Jacobian of a Hamiltonian as one sweep of the sum."""
    from oracle import pyoracle as po

    rng = np.random.default_rng(n)
    ops = [("RY", [w], [float(rng.normal())], False) for w in range(n)]
    for k in range(14):
        w = [int(x) for x in rng.permutation(n)[:4]]
        name, arity = [("DoubleExcitation", 4), ("SingleExcitation", 2), ("IsingXX", 2), ("IsingYY", 2), ("SWAP", 2),
                       ("CSWAP", 3), ("CNOT", 2)][k % 7]
        ops.append((name, w[:arity], [float(rng.normal())] if "SWAP" not in name and name != "CNOT" else [],
                    bool(rng.integers(2))))
    ops += [("RX", [0], [0.3], False), ("DoubleExcitation", [0, n - 1, 1, n - 2], [0.4], False)]
    psi = po.apply_ops(n, po.zero_state(n), ops)
    terms = [qc.PauliX(0) @ qc.PauliY(n - 1), qc.PauliZ(2) @ qc.PauliZ(3), qc.PauliY(1), qc.Identity(0)]
    words, wires, coeffs = ["XY", "ZZ", "Y", "I"], [[0, n - 1], [2, 3], [1], [0]], [0.7, -1.1, 0.25, 2.0]
    h = np.zeros_like(psi)
    for word, ws, c in zip(words, wires, coeffs):
        h = h + c * po.apply_ops(n, psi, [("Pauli" + p, [w], [], False) for p, w in zip(word, ws) if p != "I"])
    for trainable in (None, [0, n, n + 3, n + 9]):
        count = sum(1 for o in ops if o[2])
        tape = qc.QuantumTape([qc.Adjoint(qc.Operation(o[0], o[1], o[2])) if o[3] else qc.Operation(o[0], o[1], o[2])
                               for o in ops], [qc.expval(qc.Hamiltonian(coeffs, terms)), qc.expval(qc.PauliZ(0))],
                              trainable_params=trainable)
        tp = list(range(count)) if trainable is None else trainable
        bras = [h, po.apply_ops(n, psi, [("PauliZ", [0], [], False)])]
        ref = po.adjoint_jacobian(n, psi, bras, ops, tp)
        dev = LightningGPU(n)
        np.testing.assert_allclose(np.array(dev.adjoint_jacobian(tape)), ref, atol=1e-12, rtol=0)
        np.testing.assert_allclose(dev.state, psi, atol=1e-13, rtol=0)
        single = LightningGPU(n, c_dtype=np.complex64)
        np.testing.assert_allclose(np.array(single.adjoint_jacobian(tape)), ref, atol=2e-5, rtol=0)
