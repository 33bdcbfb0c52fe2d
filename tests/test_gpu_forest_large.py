"""Forests whose members take several workgroups for their boxes (8,192 bodies
a part) and whose dense cores put hundreds of bodies in one 30-bit cell: each
member, between small ones, has the bits it has alone."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (5, 8192, 8193, 1, 16384, 16385, 300, 70000)


@pytest.mark.parametrize("solver", ["LINEAR_BVH", "BARNES_HUT"])
@pytest.mark.parametrize("core", [1.0, 0.004])
def test_members_equal_alone(nbg, gpu_ctx, solver, core):
    p = nbg.default_params()
    p.solver, p.theta, p.leaf_size, p.morton_bits, p.eps2 = getattr(nbg, solver), 0.7, 16, 30, 1e-4
    p.sum_mode = nbg.SUM_FAST
    sets = []
    for k, n in enumerate(SIZES):
        b = nbg.plummer(n, seed=60 + k)
        for a in (b.x, b.y, b.z):
            a[n // 10:] *= np.float32(core)  # most bodies in a few cells
            a += np.float32(k - 3)           # boxes that share no side
        sets.append(b)
    batch = nbg.Batch(gpu_ctx, sum(SIZES), len(SIZES), sum_mode=nbg.SUM_FAST)
    ids = [batch.add(p, b) for b in sets]
    batch.update_accelerations()
    for i, b in zip(ids, sets):
        _, got = batch.get(i, accelerations=True)
        s = nbg.System(gpu_ctx, p, b.n)
        s.set_state(b)
        want = s.update_accelerations()
        s.close()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), b.n
    batch.close()


@pytest.mark.parametrize("solver", ["LINEAR_BVH", "BARNES_HUT"])
@pytest.mark.parametrize("mode", ["SUM_FAST", "SUM_ORDERED"])
def test_turns_of_the_walk(nbg, gpu_ctx, solver, mode):
    """Workgroups of several whole turns of the XCDs and a rest, members of
    different angles: every target is walked, with the bits it has alone."""
    sizes, angles = (40000, 70001, 3, 30000), (1.0, 0.6, 0.5, 0.8)
    prms = []
    for t in angles:
        p = nbg.default_params()
        p.solver, p.theta, p.leaf_size, p.morton_bits, p.eps2 = getattr(nbg, solver), t, 16, 30, 1e-4
        p.sum_mode = getattr(nbg, mode)
        prms.append(p)
    sets = [nbg.plummer(n, seed=80 + n) for n in sizes]
    batch = nbg.Batch(gpu_ctx, sum(sizes), len(sizes), sum_mode=getattr(nbg, mode))
    ids = [batch.add(p, b) for p, b in zip(prms, sets)]
    batch.update_accelerations()
    for i, p, b in zip(ids, prms, sets):
        _, got = batch.get(i, accelerations=True)
        s = nbg.System(gpu_ctx, p, b.n)
        s.set_state(b)
        want = s.update_accelerations()
        s.close()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), b.n
    batch.close()
