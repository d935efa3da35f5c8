"""Timed cases: what a program that uses this package has it do.

Each case runs through a public entry point: the ``LightningGPU`` device, the
pybind11 module ``lightning_gpu_qubit_ops`` that a device class drives, the
``_native`` handles, or the torch layer.  Sizes are those of the benchmark
configurations and of the tests (circuit families of ``workloads.py``), or
generic.  ``exact`` restates every result in 64 bits with plain torch.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pennylane-lightning-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from pennylane_lightning_gpu import _native as N  # noqa: E402
from pennylane_lightning_gpu import circuit as qc  # noqa: E402
from pennylane_lightning_gpu import workloads as W  # noqa: E402

_DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # The smallest whole call: the 12-qubit configuration (forward, <Z_w>
        # on every wire, 12 x 144 Jacobian), one step of a small variational
        # program; bound by launches and latency.
        {"name": "step_ring_12q", "kind": "step", "family": "ring", "n": 12, "layers": 4, "obs": "all", "c64": False},
        # The headline configuration: forward and 1 x 336 Jacobian of <Z0 Z27>
        # on 28 qubits, a state of 4 GiB.
        {"name": "step_brick_28q", "kind": "step", "family": "brick", "n": 28, "layers": 6, "obs": "pair",
         "c64": False},
        # The same training step in single precision at an ordinary size.
        {"name": "step_brick_24q_c64", "kind": "step", "family": "brick", "n": 24, "layers": 6, "obs": "pair",
         "c64": True},
        # The published adjoint workload: StronglyEntanglingLayers with <Z_w>
        # on every wire, one reverse sweep per observable.
        {"name": "step_sel_23q", "kind": "step", "family": "sel", "n": 23, "layers": 2, "obs": "all", "c64": False},
        # A device execution: the 760-gate ladder circuit on 24 qubits, the
        # energy of a 256-word Hamiltonian and a marginal distribution.
        {"name": "device_ladder_24q", "kind": "device", "n": 24, "layers": 8, "terms": 256, "marginal": 10,
         "c64": False},
        # A chemistry-style energy and gradient on the device: excitation
        # gates between occupied and virtual wires, a Hamiltonian of Pauli
        # words.
        {"name": "excitations_18q", "kind": "excitations", "n": 18, "singles": 16, "doubles": 32, "terms": 64,
         "c64": False},
        # The batched configuration: 4096 circuits of 8 to 20 qubits, <Z0> and
        # its gradient for each, replayed from a plan.
        {"name": "batch_4096", "kind": "batch", "circuits": 4096, "lo": 8, "hi": 20, "layers": 3, "c64": False},
        # One training step of the torch layer: forward and backward of 256
        # circuits of 12 qubits.
        {"name": "torch_256x12q", "kind": "torch", "circuits": 256, "n": 12, "layers": 3, "c64": False},
        # Shots: 10^6 seeded samples of a 24-qubit state.
        {"name": "sample_24q", "kind": "sample", "n": 24, "shots": 1000000, "c64": False},
        # Marginal probabilities of every other wire of a 24-qubit state.
        {"name": "probs_24q", "kind": "probs", "n": 24, "wires": 10, "c64": False},
        # <H> of the 20-qubit transverse-field Ising chain as a resident CSR.
        {"name": "csr_20q", "kind": "csr", "n": 20, "c64": False},
        # Explicit matrices: a unitary on several wires, as QubitUnitary gives,
        # and a Hermitian on up to 13 wires, as the device gives for a small
        # Hamiltonian.
        {"name": "matrix_20q", "kind": "matrix", "n": 20, "gate_wires": 6, "obs_wires": 9, "c64": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "device", "excitations", "batch", "torch", "sample", "probs", "csr", "matrix"])
    c64 = rng.random() < 0.4
    if kind == "step":
        obs = rng.choice(["all", "pair"])
        n = rng.randint(8, 22 if obs == "all" else 27)
        layers = rng.randint(1, 6 if n <= 20 or obs == "pair" else 2)
        return {"kind": kind, "family": rng.choice(["ring", "brick", "sel"]), "n": n, "layers": layers, "obs": obs,
                "c64": c64}
    if kind == "device":  # 14 wires and more: Hamiltonians as Pauli words
        n = rng.randint(14, 24)
        return {"kind": kind, "n": n, "layers": rng.randint(1, 8), "terms": _log_int(rng, 8, 256),
                "marginal": rng.randint(1, 12), "c64": c64}
    if kind == "excitations":
        n = 2 * rng.randint(7, 11)
        return {"kind": kind, "n": n, "singles": rng.randint(2, 32), "doubles": rng.randint(2, 48),
                "terms": _log_int(rng, 8, 128), "c64": c64}
    if kind == "batch":
        lo = rng.randint(6, 14)
        hi = rng.randint(lo, 18)
        return {"kind": kind, "circuits": _log_int(rng, 16, 3000), "lo": lo, "hi": hi, "layers": rng.randint(1, 3),
                "c64": c64}
    if kind == "torch":
        n = rng.randint(4, 15)
        return {"kind": kind, "circuits": _log_int(rng, 8, 1024), "n": n, "layers": rng.randint(1, 3), "c64": c64}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(6, 26), "shots": _log_int(rng, 100, 1000000), "c64": c64}
    if kind == "probs":
        n = rng.randint(8, 26)
        return {"kind": kind, "n": n, "wires": rng.randint(1, min(n, 20)), "c64": c64}
    if kind == "csr":
        return {"kind": kind, "n": rng.randint(10, 20), "c64": c64}
    n = rng.randint(12, 22)
    return {"kind": "matrix", "n": n, "gate_wires": rng.randint(1, 8), "obs_wires": rng.randint(1, 10), "c64": c64}


# ------------------------------------------------------------------ inputs


def _dtype(case):
    return np.complex64 if case["c64"] else np.complex128


def _suffix(case):
    return "C64" if case["c64"] else "C128"


def _circuit(case, seed):
    make = {"ring": W.layered_ring, "brick": W.ry_rz_cz_brick, "sel": W.strongly_entangling, "ladder": W.ladder}
    return make[case.get("family", "ladder")](case["n"], case["layers"], seed=seed)


def _random_state(n, seed):
    """Normalised complex Gaussian amplitudes (the distribution of a deep circuit's state), complex128."""
    g = torch.Generator(device=_DEVICE).manual_seed(seed)
    v = torch.randn((1 << n, 2), generator=g, dtype=torch.float64, device=_DEVICE)
    return torch.view_as_complex(v / torch.linalg.vector_norm(v))


def _state_input(case, seed):
    """The case's input state as the program holds it: host amplitudes in the state's precision."""
    return _random_state(case["n"], seed).cpu().numpy().astype(_dtype(case))


def _hamiltonian(case, seed):
    """Random Pauli words, and a Z field on the wires that none of them touches (so that it spans every wire)."""
    words, wires, coeffs = W.random_pauli_hamiltonian(case["n"], case["terms"], seed=seed)
    rest = sorted(set(range(case["n"])) - {w for ws in wires for w in ws})
    return words + ["Z"] * len(rest), wires + [[w] for w in rest], np.concatenate([coeffs, np.full(len(rest), 0.5)])


def _pauli_observable(case, seed):
    words, wires, coeffs = _hamiltonian(case, seed)
    make = {"X": qc.PauliX, "Y": qc.PauliY, "Z": qc.PauliZ}
    terms = []
    for word, ws in zip(words, wires):
        obs = [make[p](w) for p, w in zip(word, ws)]
        terms.append(obs[0] if len(obs) == 1 else qc.Tensor(*obs))
    return qc.Hamiltonian(coeffs, terms)


def _excitation_ops(case, seed):
    """Occupied wires filled, then excitations between occupied and virtual wires with small angles."""
    rng = np.random.default_rng(seed)
    n, occ = case["n"], case["n"] // 2
    ops = [("PauliX", [w], [], False) for w in range(occ)]
    for _ in range(case["doubles"]):
        i, j = sorted(int(x) for x in rng.choice(occ, 2, replace=False))
        a, b = sorted(int(x) for x in rng.choice(np.arange(occ, n), 2, replace=False))
        ops.append(("DoubleExcitation", [i, j, a, b], [float(rng.normal() * 0.3)], False))
    for _ in range(case["singles"]):
        ops.append(("SingleExcitation", [int(rng.integers(occ)), int(rng.integers(occ, n))],
                    [float(rng.normal() * 0.3)], False))
    return ops


def _marginal_wires(case):
    n, k = case["n"], case.get("marginal", case.get("wires"))
    """Every other wire, then the ones between, in increasing order."""
    return sorted(sorted(range(n), key=lambda w: (w % 2, w))[:k])


def _batch_inputs(case, seed):
    """Widths by the case (the plan's composition), parameters by the seed."""
    widths = W.batch_widths(case["circuits"], case["lo"], case["hi"])
    rng = np.random.default_rng(seed)
    thetas = [rng.uniform(0, 2 * np.pi, 3 * w * case["layers"]) for w in widths]
    return widths, thetas


def _matrix_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n, kg, ko = case["n"], case["gate_wires"], min(case["obs_wires"], case["n"])
    d = 1 << kg
    u, _ = np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))
    d = 1 << ko
    a = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    h = (a + a.conj().T) / (4 * math.sqrt(d))
    gw = [int(x) for x in rng.choice(n, kg, replace=False)]
    ow = [int(x) for x in rng.choice(n, ko, replace=False)]
    return gw, u, ow, h


@functools.lru_cache(maxsize=1)
def _tfim(n):
    return W.tfim_csr(n)


# ------------------------------------------------------------------ prepare and run


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_step(case, seed):
    from pennylane_lightning_gpu import lightning_gpu_qubit_ops as Q

    ops = _circuit(case, seed)
    n, sfx = case["n"], _suffix(case)
    real = np.float32 if case["c64"] else np.float64
    adj = getattr(Q, "AdjointJacobianGPU_" + sfx)()
    named = getattr(Q, "NamedObsGPU_" + sfx)
    if case["obs"] == "all":
        obs = [named("PauliZ", [w]) for w in range(n)]
    else:
        obs = [getattr(Q, "TensorProdObsGPU_" + sfx)([named("PauliZ", [0]), named("PauliZ", [n - 1])])]
    names, wires = [o[0] for o in ops], [o[1] for o in ops]
    invs, params = [o[3] for o in ops], [o[2] for o in ops]
    return {"run": _run_step, "sv": getattr(Q, "LightningGPU_" + sfx)(n), "adj": adj, "obs": obs,
            "circuit": (names, wires, invs, params),
            "ops": adj.create_ops_list(names, [np.array(p, dtype=real) for p in params], wires, invs,
                                       [np.array([], dtype=_dtype(case)) for _ in ops]),
            "trainable": list(range(sum(1 for p in params if p))),
            "z": np.array([1, 0, 0, -1], dtype=_dtype(case)), "each": range(n) if case["obs"] == "all" else ()}


def _run_step(s):
    sv = s["sv"]
    sv.resetGPU(False)
    sv.apply(*s["circuit"])
    values = [sv.ExpectationValue("PauliZ", [w], [], s["z"]) for w in s["each"]]
    jac = np.asarray(s["adj"].adjoint_jacobian(sv, s["obs"], s["ops"], s["trainable"]), dtype=np.float64)
    return {"expval": np.real(np.asarray(values)).astype(np.float64) if values else None, "jac": jac}


def _to_tape(ops, measurements):
    return qc.QuantumTape([qc.Operation(name, wires, params) for name, wires, params, _ in ops], measurements)


def _prepare_device(case, seed):
    from pennylane_lightning_gpu.lightning_gpu import LightningGPU

    tape = _to_tape(_circuit(case, seed), [qc.expval(_pauli_observable(case, seed)), qc.probs(_marginal_wires(case))])
    return {"run": _run_device, "dev": LightningGPU(case["n"], c_dtype=_dtype(case)), "tape": tape}


def _run_device(s):
    energy, marginal = s["dev"].execute(s["tape"])
    return {"energy": float(energy), "probs": marginal}


def _prepare_excitations(case, seed):
    from pennylane_lightning_gpu.lightning_gpu import LightningGPU

    tape = _to_tape(_excitation_ops(case, seed), [qc.expval(_pauli_observable(case, seed))])
    return {"run": _run_excitations, "dev": LightningGPU(case["n"], c_dtype=_dtype(case)), "tape": tape}


def _run_excitations(s):
    energy = s["dev"].execute(s["tape"])
    grad = s["dev"].adjoint_jacobian(s["tape"], use_device_state=True)
    return {"energy": float(energy), "grad": np.array(grad, dtype=np.float64)}


def _prepare_batch(case, seed):
    widths, thetas = _batch_inputs(case, seed)
    tmpl = {}
    for w in sorted(set(widths)):
        ops, pidx = W.ring_template(w, case["layers"])
        tmpl[w] = N.Template(w, ops, pidx, [("Z", 0)])
    return {"run": _run_batch, "thetas": thetas, "tmpl": tmpl,
            "plan": N.BatchPlan([tmpl[w] for w in widths], grad=True, dtype=_dtype(case))}


def _run_batch(s):
    values, jacs = s["plan"].run(s["thetas"])
    return {"expval": values, "jac": np.concatenate(jacs)}


def _prepare_torch(case, seed):
    ops, pidx = W.ring_template(case["n"], case["layers"])
    tmpl = N.Template(case["n"], ops, pidx, [("Z", 0)])
    rng = np.random.default_rng(seed)
    theta = rng.uniform(0, 2 * np.pi, (case["circuits"], tmpl.num_params))
    weight = rng.normal(size=case["circuits"])
    return {"run": _run_torch, "tmpl": tmpl, "dtype": _dtype(case),
            "params": torch.tensor(theta, device="cuda", requires_grad=True),
            "weight": torch.tensor(weight, device="cuda")}


def _run_torch(s):
    from pennylane_lightning_gpu.torch_layer import batched_expval

    p = s["params"]
    p.grad = None
    out = batched_expval(p, s["tmpl"], s["dtype"])
    (out * s["weight"]).sum().backward()
    return {"expval": out.detach(), "grad": p.grad}


def _device_state(case, seed):
    return N.State(case["n"], dtype=_dtype(case)).upload(_state_input(case, seed))


def _prepare_sample(case, seed):
    return {"run": _run_sample, "psi": _device_state(case, seed), "shots": case["shots"], "seed": seed}


def _run_sample(s):
    return s["psi"].sample(s["shots"], s["seed"]).view(np.int64)


def _prepare_probs(case, seed):
    return {"run": _run_probs, "psi": _device_state(case, seed), "wires": _marginal_wires(case)}


def _run_probs(s):
    return s["psi"].probs(s["wires"])


def _prepare_csr(case, seed):
    indptr, indices, data = _tfim(case["n"])
    return {"run": _run_csr, "psi": _device_state(case, seed), "csr": N.CSR(indptr, indices, data, dtype=_dtype(case))}


def _run_csr(s):
    return s["csr"].expval(s["psi"]).real


class _Amplitudes:
    """The amplitudes of a state where they lie, for torch."""

    def __init__(self, state):
        self.state = state
        self.__cuda_array_interface__ = {
            "shape": (1 << state.n, 2), "typestr": "<f4" if state.dtype == np.complex64 else "<f8",
            "data": (state.data_ptr(), False), "version": 2}


def _prepare_matrix(case, seed):
    gw, u, ow, h = _matrix_inputs(case, seed)
    work = N.State(case["n"], dtype=_dtype(case))
    return {"run": _run_matrix, "psi": _device_state(case, seed), "work": work,
            "view": torch.as_tensor(_Amplitudes(work), device="cuda"), "gate": [("QubitUnitary", gw, [], False, u)],
            "ow": ow, "h": h}


def _run_matrix(s):
    work = s["work"].copy_from(s["psi"])
    work.apply(s["gate"])
    return {"expval": work.expval_matrix(s["ow"], s["h"]).real, "state": s["view"]}


_PREPARE = {"step": _prepare_step, "device": _prepare_device, "excitations": _prepare_excitations,
            "batch": _prepare_batch, "torch": _prepare_torch, "sample": _prepare_sample, "probs": _prepare_probs,
            "csr": _prepare_csr, "matrix": _prepare_matrix}


# ------------------------------------------------------------------ work


def work(case):
    """Bytes and operations of one pass: every state that the path goes through read and written once (a reverse
    sweep: the state and the observable's state), 8 operations per amplitude and gate, thrice that in reverse."""
    kind, amp = case["kind"], 8 if case["c64"] else 16
    if kind in ("batch", "torch"):
        widths = W.batch_widths(case["circuits"], case["lo"], case["hi"]) if kind == "batch" else \
            [case["n"]] * case["circuits"]
        dims = [(w, 1 << w) for w in widths]
        return {"bytes": sum(6.0 * amp * d for _, d in dims),
                "flops": sum(32.0 * d * 4 * w * case["layers"] for w, d in dims)}
    n = case["n"]
    dim = float(1 << n)
    S = amp * dim
    if kind == "step":
        gates = len(_circuit(case, 1))
        sweeps = n if case["obs"] == "all" else 1
        return {"bytes": 2 * S + 4 * S * sweeps, "flops": 8 * dim * gates * (1 + 2 * sweeps + 1)}
    if kind == "device":
        return {"bytes": 3 * S, "flops": 8 * dim * (len(_circuit(case, 1)) + case["terms"])}
    if kind == "excitations":
        # a single excitation turns half of the amplitudes, a double excitation an eighth of them
        turned = case["singles"] / 2 + case["doubles"] / 8
        return {"bytes": 8 * S, "flops": 8 * dim * (4 * turned + 2 * case["terms"])}
    if kind == "sample":
        return {"bytes": S + 8.0 * case["shots"], "flops": 4 * dim}
    if kind == "probs":
        return {"bytes": S + 8.0 * (1 << case["wires"]), "flops": 4 * dim}
    if kind == "csr":
        nnz = (n + 1) * dim
        return {"bytes": nnz * (amp + amp // 2) + S + amp // 2 * dim, "flops": 8 * nnz}
    kg, ko = case["gate_wires"], min(case["obs_wires"], n)
    return {"bytes": 2 * S + 2 * S + S + 16.0 * (4.0 ** kg + 4.0 ** ko),
            "flops": 8 * dim * (2.0 ** kg + 2.0 ** ko)}


# ------------------------------------------------------------------ results in 64 bits

_X = np.array([[0, 1], [1, 0]], dtype=complex)
_Y = np.array([[0, -1j], [1j, 0]])
_Z = np.diag([1.0 + 0j, -1.0])


def _rotation(p, theta):
    c, s = math.cos(theta / 2), math.sin(theta / 2)
    return c * np.eye(2) - 1j * s * p, -0.5 * s * np.eye(2) - 0.5j * c * p


def _excitation(dim, lo, hi, theta):
    c, s = math.cos(theta / 2), math.sin(theta / 2)
    u, d = np.eye(dim, dtype=complex), np.zeros((dim, dim), dtype=complex)
    u[lo, lo] = u[hi, hi] = c
    u[lo, hi], u[hi, lo] = -s, s
    d[lo, lo] = d[hi, hi] = -s / 2
    d[lo, hi], d[hi, lo] = -c / 2, c / 2
    return u, d


def _matrices(name, theta):
    """Matrix of a gate and its derivative by the gate's angle."""
    if name in ("RX", "RY", "RZ"):
        return _rotation({"RX": _X, "RY": _Y, "RZ": _Z}[name], theta)
    if name == "SingleExcitation":
        return _excitation(4, 1, 2, theta)
    if name == "DoubleExcitation":
        return _excitation(16, 3, 12, theta)
    if name == "CNOT":
        return np.kron(np.diag([1, 0]), np.eye(2)) + np.kron(np.diag([0, 1]), _X), None
    if name == "CZ":
        return np.diag([1.0 + 0j, 1, 1, -1]), None
    return {"PauliX": _X, "PauliY": _Y, "PauliZ": _Z}[name], None


def _gate(v, n, wires, mat):
    """mat on `wires` (first: most significant) of the states v[:, 2^n]; entries of mat are numbers, or one per state."""
    k = len(wires)
    order = sorted(range(k), key=lambda i: wires[i])
    shape, prev = [v.shape[0]], 0
    for i in order:
        shape += [1 << (wires[i] - prev), 2]
        prev = wires[i] + 1
    t = v.view(shape + [1 << (n - prev)])
    at = {i: 2 + 2 * j for j, i in enumerate(order)}

    def part(x, r):
        idx = [slice(None)] * x.dim()
        for i in range(k):
            idx[at[i]] = (r >> (k - 1 - i)) & 1
        return x[tuple(idx)]

    out = torch.empty_like(t)
    for r in range(1 << k):
        acc = None
        for c in range(1 << k):
            m = mat[r][c]
            if torch.is_tensor(m):
                m = m.view([-1] + [1] * (t.dim() - k - 1))
            elif m == 0:
                continue
            term = part(t, c) if not torch.is_tensor(m) and m == 1 else part(t, c) * m
            acc = term if acc is None else acc + term
        part(out, r).copy_(acc if acc is not None else torch.zeros((), dtype=out.dtype, device=out.device))
    return out.view(v.shape)


def _angles(ops, c64):
    return [(name, wires, float(np.float32(p[0])) if c64 and p else (p[0] if p else 0.0), bool(p))
            for name, wires, p, _ in ops]


def _forward(n, ops):
    v = torch.zeros((1, 1 << n), dtype=torch.complex128, device=_DEVICE)
    v[0, 0] = 1
    for name, wires, theta, _ in ops:
        v = _gate(v, n, wires, _matrices(name, theta)[0].tolist())
    return v


def _reverse(n, ops, psi, bras):
    """d<psi|O_j|psi>/d theta for bras[j] = O_j psi, by the adjoint method."""
    both, cols = torch.cat([psi, bras]), []
    for name, wires, theta, trained in reversed(ops):
        u, d = _matrices(name, theta)
        before = _gate(both, n, wires, u.conj().T.tolist())
        if trained:
            cols.append(2 * (both[1:].conj() @ _gate(before[:1], n, wires, d.tolist())[0]).real)
        both = before
    return torch.stack(cols[::-1], dim=1).cpu().numpy()


def _pauli_word(v, n, word, wires):
    for p, w in zip(word, wires):
        v = _gate(v, n, [w], {"X": _X, "Y": _Y, "Z": _Z}[p].tolist())
    return v


def _apply_hamiltonian(v, n, words, wires, coeffs):
    out = torch.zeros_like(v)
    for word, ws, c in zip(words, wires, coeffs):
        out += c * _pauli_word(v, n, word, ws)
    return out


def _marginal(p, n, wires):
    """Probabilities by the bits of `wires`, the first wire the most significant."""
    order = sorted(wires)
    shape, prev = [], 0
    for w in order:
        shape += [1 << (w - prev), 2]
        prev = w + 1
    p = p.view(shape + [1 << (n - prev)]).sum(dim=tuple(range(0, 2 * len(order) + 1, 2)))
    return p.permute([order.index(w) for w in wires]).reshape(-1)


def _reversed_bits(p):
    k = p.numel().bit_length() - 1
    return p.view([2] * k).permute(list(range(k))[::-1]).reshape(-1)


def _exact_batch(widths, thetas, layers):
    values, grads = np.zeros(len(widths)), [None] * len(widths)
    for w in sorted(set(widths)):
        members = [i for i, x in enumerate(widths) if x == w]
        per = max(1, (1 << 28) >> w)
        for lo in range(0, len(members), per):
            at = members[lo:lo + per]
            th = torch.tensor(np.stack([thetas[i] for i in at]), device=_DEVICE)
            ops, pidx = W.ring_template(w, layers)

            def mat(name, p, inverse=False):
                if p < 0:
                    return _matrices(name, 0.0)[0].tolist()
                c, s = torch.cos(th[:, p] / 2) + 0j, torch.sin(th[:, p] / 2) + 0j
                s = -s if inverse else s
                return {"RX": [[c, -1j * s], [-1j * s, c]], "RY": [[c, -s], [s, c]],
                        "RZ": [[c - 1j * s, 0], [0, c + 1j * s]]}[name]

            psi = torch.zeros((len(at), 1 << w), dtype=torch.complex128, device=_DEVICE)
            psi[:, 0] = 1
            for (name, ws, _, _), p in zip(ops, pidx):
                psi = _gate(psi, w, ws, mat(name, p))
            bra = _gate(psi, w, [0], _Z.tolist())
            values[at] = torch.linalg.vecdot(psi, bra).real.cpu().numpy()
            g = torch.zeros_like(th)
            for (name, ws, _, _), p in zip(reversed(ops), reversed(pidx)):
                if p >= 0:  # d/dtheta exp(-i theta G / 2) = -i G / 2 U
                    gen = {"RX": _X, "RY": _Y, "RZ": _Z}[name]
                    g[:, p] = torch.linalg.vecdot(bra, _gate(psi, w, ws, gen.tolist())).imag
                psi, bra = _gate(psi, w, ws, mat(name, p, True)), _gate(bra, w, ws, mat(name, p, True))
            for i, row in zip(at, g.cpu().numpy()):
                grads[i] = row
    return values, grads


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind == "step":
        if n > 25:
            return None
        ops = _angles(_circuit(case, seed), case["c64"])
        psi = _forward(n, ops)
        if case["obs"] == "all":
            bras = torch.cat([_gate(psi, n, [w], _Z.tolist()) for w in range(n)])
            return {"expval": (bras @ psi[0].conj()).real.cpu().numpy(), "jac": _reverse(n, ops, psi, bras)}
        return {"expval": None, "jac": _reverse(n, ops, psi, _pauli_word(psi, n, "ZZ", [0, n - 1]))}
    if kind == "device":
        psi = _forward(n, _angles(_circuit(case, seed), case["c64"]))
        h = _apply_hamiltonian(psi, n, *_hamiltonian(case, seed))
        return {"energy": float(torch.linalg.vecdot(psi[0], h[0]).real),
                "probs": _marginal(psi[0].abs() ** 2, n, _marginal_wires(case)).cpu().numpy()}
    if kind == "excitations":
        ops = _angles(_excitation_ops(case, seed), case["c64"])
        psi = _forward(n, ops)
        h = _apply_hamiltonian(psi, n, *_hamiltonian(case, seed))
        return {"energy": float(torch.linalg.vecdot(psi[0], h[0]).real), "grad": _reverse(n, ops, psi, h)[0]}
    if kind == "batch":
        values, grads = _exact_batch(*_batch_inputs(case, seed), case["layers"])
        return {"expval": values, "jac": np.concatenate(grads)}
    if kind == "torch":
        rng = np.random.default_rng(seed)
        theta = rng.uniform(0, 2 * np.pi, (case["circuits"], 3 * n * case["layers"]))
        weight = rng.normal(size=case["circuits"])
        values, grads = _exact_batch([n] * case["circuits"], list(theta), case["layers"])
        return {"expval": values, "grad": np.stack(grads) * weight[:, None]}
    if kind == "sample":
        return None
    psi = _random_state(n, seed)
    if case["c64"]:
        psi = psi.to(torch.complex64).to(torch.complex128)
    if kind == "probs":
        # the entry point's order: the first wire is the least significant bit
        return _reversed_bits(_marginal(psi.abs() ** 2, n, _marginal_wires(case))).cpu().numpy()
    if kind == "csr":  # H = -sum Z_i Z_{i+1} - 0.7 sum X_i
        v, total = psi[None], 0.0
        for w in range(n):
            if w + 1 < n:
                total -= float(torch.linalg.vecdot(v, _pauli_word(v, n, "ZZ", [w, w + 1])).real)
            total -= 0.7 * float(torch.linalg.vecdot(v, _gate(v, n, [w], _X.tolist())).real)
        return total
    gw, u, ow, h = _matrix_inputs(case, seed)

    def matvec(v, wires, m):
        k = len(wires)
        rest = [w for w in range(n) if w not in wires]
        t = v.view([2] * n).permute(list(wires) + rest).reshape(1 << k, -1)
        t = torch.from_numpy(np.ascontiguousarray(m)).to(v.device) @ t
        back = np.argsort(list(wires) + rest).tolist()
        return t.view([2] * n).permute(back).reshape(-1)

    out = matvec(psi, gw, u)
    value = float(torch.linalg.vecdot(out, matvec(out, ow, h)).real)
    return {"expval": value, "state": torch.view_as_real(out.contiguous())}
