"""Systems of 160,000 bodies and more take their targets in compact groups.
The order of the targets is a schedule: ORDERED walks give the oracle's bits
with it, whole and ragged last blocks, bodies in a plane and in one point,
and a forest that mixes grouped and other members gives each member the bits
it has alone."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _params(nbg, solver, mode, theta=0.8, leaf=16, bits=30):
    p = nbg.default_params()
    p.solver, p.theta, p.leaf_size, p.morton_bits, p.eps2 = getattr(nbg, solver), theta, leaf, bits, 1e-4
    p.sum_mode = mode
    return p


@pytest.mark.parametrize("solver,kind", [("LINEAR_BVH", 1), ("BARNES_HUT", 0)])
@pytest.mark.parametrize("n,shape", [(160000, "plummer"), (160001, "plane"), (161791, "point")])
def test_grouped_targets_same_bits(nbg, orc, gpu_ctx, n, shape, solver, kind):
    print(f"[targets] {solver} n={n} {shape}", flush=True)
    b = nbg.plummer(n, seed=n)
    if shape == "plane":
        b.z[:] = 0.25
    if shape == "point":  # a quarter of the bodies in 64 points, so that whole blocks have no extent
        k = n // 4
        for a in (b.x, b.y, b.z):
            a[:k] = np.repeat(a[:64], (k + 63) // 64)[:k]
    p = _params(nbg, solver, nbg.SUM_ORDERED, leaf=64 if shape == "point" else 16)
    if shape == "point":
        p.max_depth = 12
    s = nbg.System(gpu_ctx, p, n)
    s.set_state(b)
    acc = s.update_accelerations()
    at = np.arange(0, n, 251)
    t = orc.Tree(kind, b.x, b.y, b.z, b.m, theta=0.8, leaf=p.leaf_size, bits=30, eps2=1e-4, max_depth=p.max_depth)
    want = t.accel(b.x[at], b.y[at], b.z[at])
    assert np.array_equal(acc[at].view(np.uint32), np.asarray(want).view(np.uint32))
    s.close()


@pytest.mark.parametrize("solver", ["LINEAR_BVH", "BARNES_HUT"])
def test_mixed_forest_same_bits(nbg, gpu_ctx, solver):
    p = _params(nbg, solver, nbg.SUM_FAST)
    sizes = (300, 160000, 1, 170001, 5000)
    bodies = [nbg.plummer(n, seed=40 + n) for n in sizes]
    batch = nbg.Batch(gpu_ctx, sum(sizes), len(sizes), sum_mode=nbg.SUM_FAST)
    ids = [batch.add(p, b) for b in bodies]
    batch.update_accelerations()
    for i, b in zip(ids, bodies):
        _, got = batch.get(i, accelerations=True)
        s = nbg.System(gpu_ctx, p, b.n)
        s.set_state(b)
        want = s.update_accelerations()
        s.close()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), b.n
    batch.close()


@pytest.mark.parametrize("solver,n", [("BARNES_HUT", 160001), ("LINEAR_BVH", 500001)])
def test_every_target_once(nbg, gpu_ctx, solver, n):
    """All bodies of a grouped ORDERED pass have the bits of a walk without
    groups: the same points walked as passive ones, in Morton order."""
    b = nbg.plummer(n, seed=n)
    s = nbg.System(gpu_ctx, _params(nbg, solver, nbg.SUM_ORDERED, theta=1.0), n)
    s.set_state(b)
    acc = s.update_accelerations()
    want = s.accelerations_at(b.x, b.y, b.z)
    s.close()
    assert np.array_equal(acc.view(np.uint32), want.view(np.uint32))
