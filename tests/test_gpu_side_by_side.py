"""Reverse sweeps of several observables side by side: bit for bit the sweeps
one at a time (each keeps its own order of operations)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

from pennylane_lightning_gpu.workloads import layered_ring, strongly_entangling  # noqa: E402


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,standalone", [(9, False), (10, False), (13, True), (17, False)])
def test_sweeps_side_by_side_equal_single_sweeps(n, standalone, dtype):
    """Z words formed inside the sweep and observable states of any kind, with and without a gate that runs on its
    own between the fused passes (which first copies lambda), applying the circuit first as well."""
    ops = strongly_entangling(n, 1, seed=n) + ([("IsingXX", [1, n - 2], [0.7], False)] if standalone else [])
    ops = ops + layered_ring(n, 1, seed=n + 1)
    npar = sum(1 for o in ops if o[2])
    tp = list(range(1, npar, 2))
    psi = N.State(n, dtype).reset().apply(ops)
    zs = [[w] for w in range(n)] + [[0, n - 1]]
    many = N.adjoint_jacobian_zwords(psi, zs, ops, tp)
    for j, z in enumerate(zs):
        np.testing.assert_array_equal(many[j], N.adjoint_jacobian_zwords(psi, [z], ops, tp)[0])

    def bras():
        return [N.State(n, dtype).set_pauli_word_of(psi, w, [0, n - 1]) for w in ("XY", "ZZ", "YI")]

    many = N.adjoint_jacobian(psi, bras(), ops, tp)
    for j, b in enumerate(bras()):
        np.testing.assert_array_equal(many[j], N.adjoint_jacobian(psi, [b], ops, tp)[0])
    start = N.State(n, dtype).reset()
    both = N.adjoint_jacobian_zwords(start, zs[:2], ops, tp, apply_operations=True)
    one = [N.adjoint_jacobian_zwords(start, [z], ops, tp, apply_operations=True)[0] for z in zs[:2]]
    np.testing.assert_array_equal(both, one)
