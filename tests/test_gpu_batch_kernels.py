"""Batched circuits: the grid of a batch larger than two workgroups per CU."""

import sys

import numpy as np
import pytest

sys.path.insert(0, __file__.rsplit("/", 1)[0])

from test_gpu_batch import N, ring_template  # noqa: E402

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
