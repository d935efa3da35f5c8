"""Matrices on five and six wires at the sizes where the tile of the product
changes (2^18 amplitudes), applied and measured, with controls, against plain
numpy in 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")


def matvec(v, n, wires, m):
    rest = [w for w in range(n) if w not in wires]
    t = v.reshape([2] * n).transpose(list(wires) + rest).reshape(m.shape[0], -1)
    return (m @ t).reshape([2] * n).transpose(np.argsort(list(wires) + rest)).reshape(-1)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("k", [5, 6])
@pytest.mark.parametrize("n", [6, 7, 11, 18, 19])
def test_tiles_of_the_product(n, k, dtype):
    rng = np.random.default_rng(10 * n + k)
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v = (v / np.linalg.norm(v)).astype(dtype)
    x = v.astype(np.complex128)
    u, _ = np.linalg.qr(rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k)))
    # rows of 2^k products of 64-bit numbers; the result rounded to the state's precision
    tol = 2.3e-16 * 2 * (1 << k) + (1.2e-7 if dtype == np.complex64 else 0.0)
    for wires in (list(range(n - k, n)), list(range(k)), [int(w) for w in rng.permutation(n)[:k]]):
        s = N.State(n, dtype).upload(v)
        assert abs(s.expval_matrix(wires, u) - np.vdot(x, matvec(x, n, wires, u))) < 2.3e-16 * ((2 << k) + 64)
        s.apply([("QubitUnitary", wires, [], False, u)])
        np.testing.assert_allclose(s.download(), matvec(x, n, wires, u), atol=tol * np.abs(x).max() * 2, rtol=0)
