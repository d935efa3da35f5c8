"""Circuits of many rotations keep the norm: the factors that fused passes take
out of rotations, and the products of merged gates, round without a drift of
their own (complex128)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")

from pennylane_lightning_gpu.workloads import ladder  # noqa: E402


def test_fused_passes_keep_the_norm():
    """A ladder of 8 layers on 12 qubits merges to 96 products.  Rounding a product's entries once moves the norm by
    about 0.3e-16, 96 of them by 2.9e-16 rms; 16 circuits tell that from 5e-16 (four standard deviations).  Products
    in double precision drift by 8.4e-16."""
    off = []
    for seed in range(16):
        v = N.State(12).reset().apply(ladder(12, 8, seed=seed)).download().astype(np.clongdouble)
        off.append(float((v.real ** 2 + v.imag ** 2).sum() ** 0.5 - 1))
    assert np.sqrt(np.mean(np.square(off))) < 5e-16
