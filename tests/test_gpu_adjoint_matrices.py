"""The adjoint sweep over circuits with explicit matrices between the trainable
gates: a gate that runs on its own inside the sweep must leave the sweep's
partial sums, Jacobian rows and pointer tables alone, whatever scratch memory
its own width takes (7 and more wires: a buffer of rows; 9 and more: the
matrix in memory of its own)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

from oracle import pyoracle as po  # noqa: E402
from pennylane_lightning_gpu.workloads import layered_ring  # noqa: E402


def circuit(n, seed):
    rng = np.random.default_rng(seed)
    ops = [("RY", [w], [float(rng.normal())], False) for w in range(n)]
    for k in (3, 5, 7, 8, 9):
        k = min(k, n)
        u, _ = np.linalg.qr(rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k)))
        ops.append(("QubitUnitary", [int(x) for x in rng.permutation(n)[:k]], [], bool(rng.integers(2)), u))
        for w in (int(x) for x in rng.permutation(n)[:3]):
            ops.append((("RX", "RZ")[k % 2], [w], [float(rng.normal())], False))
        ops.append(("CNOT", [0, n - 1], [], False))
    return ops


@pytest.mark.parametrize("fusion", [True, False])
@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [8, 9, 13])
def test_adjoint_over_wide_matrices(n, dtype, fusion):
    """8 qubits take the unfused form in any case; one and several observables, formed by the caller and by the sweep."""
    ops = circuit(n, n)
    tp = list(range(sum(1 for o in ops if o[2])))
    ref_psi = po.apply_ops(n, po.zero_state(n), ops)
    words = [("X", [0]), ("ZY", [1, n - 1]), ("Z", [2])]
    ref_bras = [po.apply_ops(n, ref_psi, [("Pauli" + p, [w], [], False) for p, w in zip(word, ws)])
                for word, ws in words]
    ref = po.adjoint_jacobian(n, ref_psi, ref_bras, ops, tp)
    # Rounding: per gate some 2^k + 8 additions in the matrix's row, in
    # complex128 (1500 of them in all, forward and back); in complex64 the
    # amplitudes are rounded to single once or twice per gate (45 gates).
    tol = 4 * 1500 * 2.3e-16 if dtype == np.complex128 else 4 * 2 * 45 * 1.2e-7
    N.set_fusion(fusion)
    try:
        psi = N.State(n, dtype).reset().apply(ops)

        def bra(j):
            return N.State(n, dtype).set_pauli_word_of(psi, *words[j])

        one = N.adjoint_jacobian(psi, [bra(0)], ops, tp)
        many = N.adjoint_jacobian(psi, [bra(j) for j in range(3)], ops, tp)
        z = N.adjoint_jacobian_zwords(psi, [[2], [2]], ops, tp)
    finally:
        N.set_fusion(True)
    np.testing.assert_allclose(one, ref[:1], atol=tol, rtol=0)
    np.testing.assert_allclose(many, ref, atol=tol, rtol=0)
    np.testing.assert_allclose(z, ref[[2, 2]], atol=tol, rtol=0)


@pytest.mark.parametrize("nobs", [1, 3])
def test_more_trainable_gates_than_one_store(nobs):
    """450 trainable gates on 10 qubits, more than the partial sums of one store hold, with a gate that runs on its
    own in between: against the unfused sweep."""
    n = 10
    u, _ = np.linalg.qr(np.random.default_rng(1).normal(size=(8, 8)))
    ops = layered_ring(n, 9, seed=4) + [("QubitUnitary", [0, 4, 9], [], False, u)] + layered_ring(n, 6, seed=5)
    psi = N.State(n).reset().apply(ops)
    tp = list(range(sum(1 for o in ops if o[2])))
    fused = N.adjoint_jacobian_zwords(psi, [[w] for w in range(nobs)], ops, tp)
    N.set_fusion(False)
    try:
        plain = N.adjoint_jacobian_zwords(psi, [[w] for w in range(nobs)], ops, tp)
    finally:
        N.set_fusion(True)
    # 600 gates of some 8 roundings each on two states
    np.testing.assert_allclose(fused, plain, atol=2 * 8 * 600 * 2.3e-16, rtol=0)


@pytest.mark.parametrize("fusion", [True, False])
@pytest.mark.parametrize("n", [8, 14])
def test_observable_states_of_another_stream(n, fusion):
    """States that live on another stream than psi: the gates that run on their own stay in order with the sweep."""
    ops = circuit(n, n + 1)
    tp = list(range(sum(1 for o in ops if o[2])))
    stream = N.C.c_void_p()
    N.check(N.lib().lgh_stream_create(0, N.C.byref(stream)))
    N.set_fusion(fusion)
    try:
        psi = N.State(n).reset().apply(ops)
        words = [("X", [0]), ("ZY", [1, n - 1])]
        same = N.adjoint_jacobian(psi, [N.State(n).set_pauli_word_of(psi, *w) for w in words], ops, tp)
        for _ in range(5):
            other = [N.State(n, stream=stream).set_pauli_word_of(psi, *w) for w in words]
            np.testing.assert_array_equal(N.adjoint_jacobian(psi, other, ops, tp), same)
        del other
    finally:
        N.set_fusion(True)
    N.check(N.lib().lgh_stream_synchronize(stream))
    N.check(N.lib().lgh_stream_destroy(stream))
