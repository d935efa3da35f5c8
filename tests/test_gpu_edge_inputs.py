"""Sums without terms: zero, whatever the memory that takes them holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

from pennylane_lightning_gpu import lightning_gpu_qubit_ops as Q  # noqa: E402


def poisoned(n, dtype):
    bad = np.full(1 << n, complex(np.nan, np.inf), dtype=dtype)
    bad[::3] = complex(-np.inf, 1)
    return N.State(n, dtype).upload(bad)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 5, 12, 14])
def test_sum_without_terms_is_zero(n, dtype):
    src, dst = N.State(n, dtype).reset(), poisoned(n, dtype)
    fn = N.lib().lgh_sv_pauli_sum_from
    fn.argtypes = [N.C.c_void_p, N.C.c_void_p, N.C.c_int64, N.C.c_char_p] + [N.C.c_void_p] * 3
    N.check(fn(dst.handle, src.handle, 0, None, None, None, None))
    np.testing.assert_array_equal(dst.download(), np.zeros(1 << n, dtype=dtype))


@pytest.mark.parametrize("n", [3, 10])
def test_jacobian_row_of_no_terms_is_zero(n):
    """The observable state is formed in recycled memory."""
    adj = Q.AdjointJacobianGPU_C128()
    ops = adj.create_ops_list(["RX", "RY"], [np.array([0.3]), np.array([0.4])], [[0], [n - 1]], [False, False],
                              [np.array([], dtype=complex)] * 2)
    sv = Q.LightningGPU_C128(n)
    for _ in range(4):
        held = [poisoned(n, np.complex128) for _ in range(3)]
        del held
        rows = adj.adjoint_jacobian_summed(sv, [Q.NamedObsGPU_C128("PauliZ", [0])], [0, 0, 1], ops, [0, 1])
        np.testing.assert_array_equal(np.asarray(rows)[0], [0.0, 0.0])
        none = adj.adjoint_jacobian(sv, [Q.HamiltonianGPU_C128(np.array([]), [])], ops, [0, 1])
        np.testing.assert_array_equal(np.asarray(none), [[0.0, 0.0]])
