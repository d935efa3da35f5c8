"""A call that asks for more device memory than there is fails with an
out-of-memory error, and the calls after it work; sweeps side by side take a
bounded amount of memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

LGH_ERR_OUT_OF_MEMORY = 3


def test_calls_after_a_failed_workspace_request():
    """A Jacobian of 2^20 rows x 2^17 columns (1 TiB) fails before any row is formed."""
    n, rows, cols = 4, 1 << 20, 1 << 17
    ops = [("RX", [0], [0.4], False), ("RY", [3], [0.2], False)]
    psi = N.State(n).reset().apply(ops)
    before = psi.probs([0, 3])
    bra = N.State(n).set_pauli_word_of(psi, "Z", [0])
    arr, keep = N.make_ops(ops)
    handles = (N.C.c_void_p * rows)(*[bra.handle.value] * rows)
    tp = np.arange(cols, dtype=np.int64)
    jac = np.zeros(1)
    rc = N.lib().lgh_adjoint_jacobian(psi.handle, handles, rows, arr, len(ops), tp.ctypes.data, cols, 0,
                                      jac.ctypes.data)
    assert rc == LGH_ERR_OUT_OF_MEMORY, N.lib().lgh_last_error()
    np.testing.assert_array_equal(psi.probs([0, 3]), before)
    total, _ = psi.expval_pauli_words(["Z", "Z"], [[0], [3]], [1.0, 2.0])
    assert total == pytest.approx(np.cos(0.4) + 2 * np.cos(0.2), abs=1e-14)
    got = N.adjoint_jacobian(psi, [N.State(n).set_pauli_word_of(psi, "Z", [0])], ops, [0, 1])
    np.testing.assert_allclose(got, [[-np.sin(0.4), 0.0]], atol=1e-14, rtol=0)


def test_memory_of_sweeps_side_by_side():
    """300 observables of 20 qubits: what the call takes, a lambda and partial sums per sweep, stays below 2.25 GiB
    (and 64 MiB for what does not depend on the number of sweeps)."""
    n, nobs = 20, 300
    ops = [("RY", [w], [0.1 * w], False) for w in range(n)]
    psi = N.State(n, np.complex64).reset().apply(ops)
    bras = [N.State(n, np.complex64).set_pauli_word_of(psi, "Z", [j % n]) for j in range(nobs)]
    N.adjoint_jacobian(psi, bras[:1], ops, [0])  # buffers that do not grow with the sweeps
    free, total = N.C.c_uint64(), N.C.c_uint64()
    N.check(N.lib().lgh_pool_trim(0))
    N.check(N.lib().lgh_device_memory(0, N.C.byref(free), N.C.byref(total)))
    before = free.value
    jac = N.adjoint_jacobian(psi, bras[1:], ops, list(range(n)))
    N.check(N.lib().lgh_device_memory(0, N.C.byref(free), N.C.byref(total)))
    assert before - free.value <= (9 << 28) + (64 << 20)
    # observables repeat every 20 rows, within a group of sweeps and from one group to the next
    np.testing.assert_array_equal(jac[n:], jac[:-n])
    # row j: d<Z_w> / d theta_w = -sin theta_w for w = (j + 1) % 20, in single precision
    w = np.arange(1, nobs) % n
    ref = np.zeros((nobs - 1, n))
    ref[np.arange(nobs - 1), w] = -np.sin(0.1 * w)
    np.testing.assert_allclose(jac, ref, atol=20 * 1.2e-7 * 4, rtol=0)
