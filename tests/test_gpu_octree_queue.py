"""The octree's summaries on both sides of the queue's two forms (one place at
a time, or one for all of a workgroup of 1,024 bodies; quadrupoles change at
512 workgroups): sampled ORDERED accelerations have the oracle's bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quad,n", [(False, 1023), (False, 1025), (False, 20481), (True, 511 * 1024), (True, 511 * 1024 + 1)])
def test_queue_forms(nbg, orc, gpu_ctx, quad, n):
    print(f"[octree queue] n={n} quad={quad}", flush=True)
    b = nbg.plummer(n, seed=17)
    p = nbg.default_params()
    p.solver, p.theta, p.leaf_size, p.eps2 = nbg.BARNES_HUT_QUADRUPOLE if quad else nbg.BARNES_HUT, 0.9, 32, 1e-4
    p.sum_mode = nbg.SUM_ORDERED
    s = nbg.System(gpu_ctx, p, n)
    s.set_state(b)
    acc = s.update_accelerations()
    at = np.arange(0, n, max(1, n // 400))
    t = orc.Tree(3 if quad else 0, b.x, b.y, b.z, b.m, theta=0.9, leaf=32, max_depth=p.max_depth, eps2=1e-4)
    want = np.asarray(t.accel(b.x[at], b.y[at], b.z[at]))
    assert np.array_equal(acc[at].view(np.uint32), want.view(np.uint32))
    s.close()


@pytest.mark.parametrize("quad,n", [(False, 128 * 1024), (False, 128 * 1024 + 1), (True, 192 * 1024 + 1),
                                    (False, 129 * 64 * 1024 + 1)])
def test_segments(nbg, orc, gpu_ctx, quad, n):
    """As many segments of 1,024 bodies as the last workgroup joins, one more,
    a middle pass whose last workgroup owns one body, and two middle passes."""
    test_queue_forms(nbg, orc, gpu_ctx, quad, n)
