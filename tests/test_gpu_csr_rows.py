"""Sparse matrices whose rows differ in length: the rule that picks a kernel by
the longest row, each kernel with and without an output state, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")


def matrix(n, kind, rng):
    rows = 1 << n
    length = {"even": np.full(rows, 5), "dense row": np.where(np.arange(rows) == rows // 3, rows, 1),
              "dense last": np.where(np.arange(rows) == rows - 1, rows, 0),
              "some long": np.where(np.arange(rows) % 64 == 5, min(rows, 700), 3),
              "empty": np.zeros(rows, dtype=int)}[kind]
    indptr = np.concatenate([[0], np.cumsum(length)]).astype(np.int64)
    nnz = int(indptr[-1])
    return indptr, rng.integers(0, rows, nnz), rng.normal(size=nnz) + 1j * rng.normal(size=nnz)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [3, 7, 11, 15])
@pytest.mark.parametrize("kind", ["even", "dense row", "dense last", "some long", "empty"])
def test_rows_of_any_length(n, kind, dtype):
    rng = np.random.default_rng(n)
    indptr, cols, vals = matrix(n, kind, rng)
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v = (v / np.linalg.norm(v)).astype(dtype)
    vals = vals.astype(dtype).astype(np.complex128)
    x = v.astype(np.complex128)
    y, bound = np.zeros(1 << n, dtype=complex), np.zeros(1 << n)
    row = np.repeat(np.arange(1 << n), np.diff(indptr))
    np.add.at(y, row, vals * x[cols])
    np.add.at(bound, row, 2 * np.abs(vals * x[cols]))
    m = N.CSR(indptr, cols, vals, dtype=dtype)
    psi, out = N.State(n, dtype).upload(v), N.State(n, dtype)
    m.apply(out, psi)
    # a row of k entries: k products and sums in 64 bits, the result rounded to the state's precision
    eps = 2.3e-16 * (np.diff(indptr) + 4)
    single = 1.2e-7 if dtype == np.complex64 else 0.0
    assert np.all(np.abs(out.download() - y) <= eps * bound + single * np.abs(y) + 1e-30)
    assert abs(m.expval(psi) - np.vdot(x, y)) <= (eps * bound * np.abs(x)).sum() + 2.3e-16 * (1 << n) * np.abs(x * y).sum()
