"""Edges of the measurement kernels: tiles, splits, remainders and the sizes
at which a rule changes the route.  Each result is compared with plain numpy
in 64 bits on the amplitudes that the state holds (complex64 states are read
in single precision and summed in double, so the same bounds hold)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("pennylane_lightning_gpu._native")


def rand_state(n, seed, dtype=np.complex128):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return (v / np.linalg.norm(v)).astype(dtype)


def np_probs(psi, n, wires):
    """wires[0] is the least significant output bit."""
    p = np.abs(psi.astype(np.complex128)) ** 2
    idx = np.arange(1 << n)
    out = np.zeros(1 << n, dtype=np.int64)
    for j, w in enumerate(wires):
        out |= ((idx >> (n - 1 - w)) & 1) << j
    return np.bincount(out, weights=p, minlength=1 << len(wires))


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 4, 6, 7, 9, 13, 18, 21])
def test_probs_edges(n, dtype):
    """No wire, one, the lanes' own, the highest, all; 13, 14 and more output
    wires (the lanes change their index bits at 14); scrambled orders."""
    psi = rand_state(n, 3 * n, dtype)
    s = N.State(n, dtype).upload(psi)
    rng = np.random.default_rng(n)
    for k in sorted({0, 1, 2, n // 2, n - 1, n, 5, 6, 8, 10, 11, 13, 14, 16}):
        if k < 0 or k > min(n, 18):
            continue
        for wires in (list(range(k)), list(range(n - k, n)), [int(x) for x in rng.permutation(n)[:k]]):
            # sums of up to 2^n rounded positive terms: relative error below 2^n eps
            np.testing.assert_allclose(s.probs(wires), np_probs(psi, n, wires), rtol=max(1e-14, 2.0 ** n * 2.3e-16),
                                       atol=0, err_msg=f"n={n} wires={wires}")


def concentrated(n, seed):
    """Few large amplitudes: a tile (2^11 amplitudes) that takes most shots, one amplitude that takes a third of
    them, zero tiles at both ends where there is room."""
    psi = rand_state(n, seed)
    psi[(1 << n) // 3] = 0.8
    if n >= 13:
        psi[:2048] = psi[-2048:] = 0
        psi[2048 * 2:2048 * 3] *= 10
    return psi / np.linalg.norm(psi)


@pytest.mark.parametrize("n", [1, 6, 10, 11, 12, 15, 17])
@pytest.mark.parametrize("shots", [1, 63, 4096, 4097, 30000])
def test_sampler_tiles_bit_exact(n, shots):
    """Spread and concentrated states (a tile of more than 4096 shots is shared by several workgroups), a basis
    state, and an unnormalised state, against the oracle's inverse CDF; samples are whole numbers and stay equal."""
    from oracle import pyoracle as po

    basis = np.zeros(1 << n, dtype=np.complex128)
    basis[(1 << n) * 2 // 3] = 1
    for k, psi in enumerate((rand_state(n, n), concentrated(n, n + 1), basis, 0.3 * rand_state(n, n + 2))):
        for dtype in (np.complex128, np.complex64):
            p = psi.astype(dtype)
            got = N.State(n, dtype).upload(p).sample(shots, 77 + k)
            np.testing.assert_array_equal(got, po.sample(n, p, shots, 77 + k), err_msg=f"state {k} {dtype}")


def test_sampling_a_zero_state_is_an_error():
    s = N.State(12)
    s.upload(np.zeros(1 << 12, dtype=np.complex128))
    with pytest.raises(N.LghError, match="zero state"):
        s.sample(100, 1)
    with pytest.raises(N.LghError, match="zero state"):
        s.sample_bits(100, 1)
