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


def np_matrix(psi, n, wires, m, ctrl=()):
    """m on `wires` (first: most significant) where the control wires are 1."""
    k = len(wires)
    rest = [w for w in range(n) if w not in wires and w not in ctrl]
    order = list(ctrl) + list(wires) + rest
    t = np.ascontiguousarray(psi.astype(np.complex128).reshape([2] * n).transpose(order)).reshape(1 << len(ctrl),
                                                                                               1 << k, -1)
    t[-1] = m @ t[-1]
    return t.reshape([2] * n).transpose(np.argsort(order)).reshape(-1)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,k", [(4, 4), (5, 4), (9, 4), (13, 4), (5, 5), (6, 5), (9, 5), (13, 5), (6, 6), (11, 6), (14, 6), (7, 7), (12, 7), (15, 7),
                                 (9, 8), (14, 8), (10, 10), (16, 10)])
def test_dense_matrices_on_many_wires(n, k, dtype):
    """Matrix gates and expectations on four and more wires: one group, fewer groups than a tile's columns, tiles
    and remainders; the lowest wires, the highest, scattered ones in a scrambled order; controls; the adjoint.
    Products of 2^k terms of unitary rows: error below 2^(k/2 + 2) eps of the amplitudes' scale."""
    rng = np.random.default_rng(100 * n + k)
    psi = rand_state(n, n + k, dtype)
    D = 1 << k
    u, _ = np.linalg.qr(rng.normal(size=(D, D)) + 1j * rng.normal(size=(D, D)))
    eps = np.finfo(np.float64 if dtype == np.complex128 else np.float32).eps
    tol = 4 * np.sqrt(D) * eps
    for wires in (list(range(k)), list(range(n - k, n)), [int(x) for x in rng.permutation(n)[:k]]):
        s = N.State(n, dtype).upload(psi)
        # not Hermitian: both parts of the value; evaluated in double for complex64 states as well
        ev = s.expval_matrix(wires, u)
        assert abs(ev - np.vdot(psi.astype(np.complex128), np_matrix(psi, n, wires, u))) < 4 * np.sqrt(D) * 2.3e-16
        s.apply([("QubitUnitary", wires, [], False, u)])
        np.testing.assert_allclose(s.download(), np_matrix(psi, n, wires, u), atol=tol, rtol=0)
        s.apply([("QubitUnitary", wires, [], True, u)])
        np.testing.assert_allclose(s.download(), psi, atol=2 * tol, rtol=0)


@pytest.mark.parametrize("n,k,ctrl", [(5, 4, 1), (12, 4, 3), (7, 5, 1), (12, 5, 2), (13, 6, 1), (12, 7, 2), (16, 7, 1)])
def test_controlled_dense_matrices_on_many_wires(n, k, ctrl):
    rng = np.random.default_rng(n + k)
    psi = rand_state(n, n + k)
    D = 1 << k
    u, _ = np.linalg.qr(rng.normal(size=(D, D)) + 1j * rng.normal(size=(D, D)))
    w = [int(x) for x in rng.permutation(n)[:k + ctrl]]
    arr, keep = N.make_ops([("QubitUnitary", w, [], False, u)])
    arr[0].num_ctrl = ctrl
    s = N.State(n).upload(psi)
    N.check(N.lib().lgh_apply(s.handle, arr, 1))
    np.testing.assert_allclose(s.download(), np_matrix(psi, n, w[ctrl:], u, w[:ctrl]),
                               atol=4 * np.sqrt(D) * 2.3e-16, rtol=0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [2, 7, 9, 11, 12, 13, 16])
def test_pauli_words_by_flip_mask(n, dtype):
    """States smaller than, equal to and larger than a tile (2^12 amplitudes); many words of one flip mask (a launch
    holds 64 words, a wavefront 8 of them), Z words up to the one on every wire (every tile bit signed), flips on
    every wire, every number of Y factors."""
    rng = np.random.default_rng(n)
    psi = rand_state(n, 5 * n, dtype)
    every = list(range(n))
    words, wires = ["Z" * n, "X" * n, "Y" * n, "", "I"], [every, every, every, [], [0]]
    for k in range(80):  # Z words
        ws = [int(x) for x in rng.permutation(n)[:int(rng.integers(1, n + 1))]]
        words.append("Z" * len(ws))
        wires.append(ws)
    for k in range(90):  # few masks, many words of each
        ws = [int(x) for x in rng.permutation(n)[:int(rng.integers(1, min(n, 6) + 1))]]
        letters = ["XY"[int(rng.integers(2))] if w < min(n, 3) else "Z" for w in ws]
        words.append("".join(letters))
        wires.append(ws)
    for k in range(90):
        ws = [int(x) for x in rng.permutation(n)[:int(rng.integers(1, min(n, 4) + 1))]]
        words.append("".join(rng.choice(list("XYZI"), len(ws))))
        wires.append(ws)
    total, per = N.State(n, dtype).upload(psi).expval_pauli_words(words, wires, np.arange(len(words)) * 0.01)
    p = psi.astype(np.complex128)
    idx = np.arange(1 << n)
    ref = []
    for word, ws in zip(words, wires):
        flip = sum(1 << (n - 1 - w) for c, w in zip(word, ws) if c in "XY")
        zy = sum(1 << (n - 1 - w) for c, w in zip(word, ws) if c in "YZ")
        par = np.array([bin(int(i) & zy).count("1") & 1 for i in idx]) if n <= 9 else \
            np.bitwise_count(idx & zy).astype(np.int64) & 1
        ref.append(np.real(1j ** word.count("Y") * np.sum((1 - 2 * par) * np.conj(p[idx ^ flip]) * p)))
    # sums of 2^n products of total size 1
    np.testing.assert_allclose(per, ref, atol=2.0 ** (n / 2) * 4e-16, rtol=0)
    np.testing.assert_allclose(total, np.dot(np.arange(len(words)) * 0.01, ref), atol=2.0 ** (n / 2) * 4e-14, rtol=0)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,avg", [(1, 1), (5, 3), (8, 6), (9, 7), (9, 12), (9, 13), (10, 24), (10, 25), (10, 47),
                                   (11, 60)])
@pytest.mark.parametrize("shape", ["even", "ragged", "one_long"])
def test_csr_rows_of_every_length(n, avg, shape, dtype):
    """<H> and H|x> with rows on both sides of each change of the number of
    lanes per row: rows of one length, rows of 0 to twice the average, and one
    row that runs over several steps of its workgroup among empty ones.  Sums
    in double: relative to the sum of magnitudes, at most 2^16 terms of
    2^-53 each, 1e-11; H|x> in complex64 is rounded once more (2^-24)."""
    rng = np.random.default_rng(1000 * n + avg)
    D = 1 << n
    if shape == "even":
        cnt = np.full(D, avg)
    elif shape == "ragged":
        cnt = rng.integers(0, 2 * avg + 1, D)
    else:
        cnt = np.zeros(D, dtype=np.int64)
        cnt[D // 3] = avg * D
    ip = np.zeros(D + 1, dtype=np.int64)
    np.cumsum(cnt, out=ip[1:])
    ix = rng.integers(0, D, ip[-1])
    d = (rng.normal(size=ip[-1]) + 1j * rng.normal(size=ip[-1])).astype(dtype)
    v = rng.normal(size=D) + 1j * rng.normal(size=D)
    v = (v / np.linalg.norm(v)).astype(dtype)
    H, x = N.CSR(ip, ix, d, dtype=dtype), N.State(n, dtype)
    x.upload(v)
    row = np.repeat(np.arange(D), cnt)
    terms = d.astype(np.complex128) * v.astype(np.complex128)[ix]
    y = np.bincount(row, terms.real, D) + 1j * np.bincount(row, terms.imag, D)
    mag = np.bincount(row, np.abs(terms), D)
    e = H.expval(x)
    ref = np.vdot(v.astype(np.complex128), y)
    assert abs(e - ref) <= 1e-11 * max(np.sum(np.abs(v) * mag), 1e-300)
    out = N.State(n, dtype)
    H.apply(out, x)
    tol = 1e-11 if dtype == np.complex128 else 1e-11 + 2.0**-23
    assert np.all(np.abs(out.download() - y) <= tol * np.maximum(mag, 1e-300))
