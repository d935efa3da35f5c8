"""Gates that mix pairs of basis states at the sizes and bits where their route
changes between the pairs' kernels and the matrix kernels, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

from oracle import pyoracle as po  # noqa: E402

GATES = [("SWAP", 0), ("IsingXX", 1), ("IsingYY", 1), ("SingleExcitation", 1), ("CSWAP", 0)]


def pairs_of_bits(n):
    return [(low, high) for low in range(5) for high in (low + 1, n - 1)]


def smooth_state(n, dtype):
    v = np.exp(1j * 0.37 * np.arange(1 << n)) * (1 + np.arange(1 << n) % 7)
    return (v / np.linalg.norm(v)).astype(dtype)


@pytest.mark.parametrize("n,dtype", [(22, np.complex64), (23, np.complex64), (22, np.complex128)])
def test_forward_routes(n, dtype):
    """The bits on both sides of a line of 64 bytes; complex64 changes at 64 MiB (23 qubits)."""
    psi = smooth_state(n, dtype)
    ops = []
    for i, (low, high) in enumerate(pairs_of_bits(n)):
        for name, p in GATES:
            ws = ([n // 2] if name == "CSWAP" else []) + [n - 1 - high, n - 1 - low][::1 if i % 2 else -1]
            ops.append((name, ws, [0.2 + 0.1 * i] * p, bool(i % 3 == 0)))
    s = N.State(n, dtype).upload(psi)
    for op in ops:
        s.apply([op])
    ref = po.apply_ops(n, psi.astype(np.complex128), ops)
    # 50 gates of two products and a sum each, amplitudes below 4e-3 (norm 1 spread over the state)
    eps = 1.2e-7 if dtype == np.complex64 else 2.3e-16
    np.testing.assert_allclose(s.download(), ref, atol=50 * 4 * eps * np.abs(ref).max(), rtol=0)


@pytest.mark.parametrize("n,dtype", [(21, np.complex64), (22, np.complex64), (21, np.complex128)])
def test_adjoint_routes(n, dtype):
    """32 MiB (22 qubits in complex64, 21 in complex128) and the size below."""
    ops = [("RY", [w], [0.3 + 0.1 * w], False) for w in range(0, n, 5)]
    for i, (low, high) in enumerate(pairs_of_bits(n)):
        name, p = GATES[i % 4]
        ops.append((name, [n - 1 - high, n - 1 - low], [0.2 + 0.1 * i] * p, bool(i % 2)))
    ops.append(("CSWAP", [3, 0, n - 1], [], False))
    tp = list(range(sum(1 for o in ops if o[2])))
    psi0 = po.zero_state(n)
    psi0[:] = smooth_state(n, np.complex128)
    ref_psi = po.apply_ops(n, psi0, ops)
    word = ("XZ", [0, n - 1])
    bra = po.apply_ops(n, ref_psi, [("PauliX", [0], [], False), ("PauliZ", [n - 1], [], False)])
    ref = po.adjoint_jacobian(n, ref_psi, [bra], ops, tp)
    psi = N.State(n, dtype).upload(smooth_state(n, dtype)).apply(ops)
    got = N.adjoint_jacobian(psi, [N.State(n, dtype).set_pauli_word_of(psi, *word) for _ in range(2)], ops, tp)
    # 16 gates forward and back on two states of norm 1
    tol = 2 * 2 * 16 * 4 * (1.2e-7 if dtype == np.complex64 else 2.3e-16)
    np.testing.assert_allclose(got, np.concatenate([ref, ref]), atol=tol, rtol=0)
