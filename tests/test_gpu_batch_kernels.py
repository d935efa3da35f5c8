"""Batched circuits: the grid of a batch larger than two workgroups per CU,
and rotations whose cosines are taken out of the gates."""

import sys

import numpy as np
import pytest

sys.path.insert(0, __file__.rsplit("/", 1)[0])

from test_gpu_batch import N, oracle_run, ring_template  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("count", [1, 512, 513, 1100])
def test_batches_over_two_workgroups_per_cu(dtype, count):
    """Every circuit is computed by one workgroup whatever the grid: the
    results of a large batch equal those of batches of one, bit for bit, from
    the eager launch and from a tuned plan."""
    rng = np.random.default_rng(count)
    widths = [3, 8, 9, 11]
    tm = {w: N.Template(w, *ring_template(w, layers=2), [("Z", 0)]) for w in widths}
    ts = [tm[widths[k % 4]] for k in range(count)]
    thetas = [rng.uniform(0, 2 * np.pi, t.num_params) for t in ts]
    ev, jac = N.batch_run(ts, thetas, dtype=dtype)
    plan = N.BatchPlan(ts, grad=True, dtype=dtype)
    assert plan.info()["grid_per_cu"] in ((1, 2) if count <= 512 else (1, 2, 3))
    for _ in range(2):
        ev_p, jac_p = plan.run(thetas)
        np.testing.assert_array_equal(ev_p, ev)
        for x, y in zip(jac_p, jac):
            np.testing.assert_array_equal(x, y)
    plan.close()
    for c in sorted({0, count // 2, count - 1}):
        e1, j1 = N.batch_run([ts[c]], [thetas[c]], dtype=dtype)
        assert e1[0] == ev[c]
        np.testing.assert_array_equal(j1[0], jac[c])


@pytest.mark.parametrize("angles", ["random", "pi", "near_pi", "zero", "large"])
@pytest.mark.parametrize("n,layers,gates", [
    (3, 2, ("RX", "RY", "RZ")),    # padded tile
    (9, 14, ("RX", "RY", "RZ")),   # one tile, several groups of passes
    (10, 3, ("RZ", "RY", "RZ")),
    (10, 2, ("RY",)),              # real gates only
    (8, 60, ("RX", "RX")),         # products below a pass's floor
])
def test_rotations_with_their_cosines_taken_out(n, layers, gates, angles):
    """Expectation values and gradients against the oracle: half angles at
    and near pi/2 (cosines of 6e-17 and 1e-13), products that reach the floor
    within a pass, deep circuits, inverse gates.  Values of order one; at most
    2500 gate applications of 4 roundings each: 2500 * 4 * 2^-53 = 1.1e-12, and
    a factor of 10 for the sums."""
    rng = np.random.default_rng(n * layers)
    ops, pidx, k = [], [], 0
    for _ in range(layers):
        for w in range(n):
            for g in gates:
                ops.append((g, [w], [0.0], k % 3 == 0))
                pidx.append(k)
                k += 1
        for w in range(n):
            ops.append(("CNOT", [w, (w + 1) % n], [], False))
            pidx.append(-1)
    theta = rng.uniform(0, 2 * np.pi, k)
    if angles == "pi":
        theta[:] = np.pi
    elif angles == "near_pi":
        theta[::2] = np.pi * (1 + 1e-13)
    elif angles == "zero":
        theta[:] = 0.0
    elif angles == "large":
        theta *= 1e3
    obs = [("X", 0)] if n == 9 else [("Z", 0), ("Y", n - 1)]
    ev, jac = N.batch_run([N.Template(n, ops, pidx, obs)], [theta])
    ref, jref = oracle_run(n, ops, pidx, theta, obs)
    assert abs(ev[0] - ref) <= 1e-11
    np.testing.assert_allclose(jac[0], jref, rtol=0, atol=1e-11)
