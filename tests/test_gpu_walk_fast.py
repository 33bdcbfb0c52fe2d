"""The FAST walks at the edges of their schedule: target groups that end
inside a wave, leaves of more than a row and of more than a wave of bodies,
stacks that fill up (small opening angles, leaves of one body), and every
number of waves per group.  Interaction counts equal the oracle's, and
accelerations agree within 1e-5 of max(|a|, a_rms), the bound of the FAST
mode."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FAST_TOL = 1e-5
SOLVERS = {"lbvh": 1, "octree": 0, "lbvh4p": 4, "octree4p": 3}


def _params(nbg, solver, theta, leaf, eps2):
    p = nbg.default_params()
    p.solver, p.theta, p.leaf_size, p.eps2, p.sum_mode = SOLVERS[solver], theta, leaf, eps2, nbg.SUM_FAST
    return p


def _check(got, want):
    mag = np.linalg.norm(want, axis=1)
    floor = max(float(np.sqrt(np.mean(mag ** 2))), 1e-30)
    assert float(np.max(np.linalg.norm(got - want, axis=1) / np.maximum(mag, floor))) <= FAST_TOL


@pytest.mark.parametrize("solver", list(SOLVERS))
@pytest.mark.parametrize("n,leaf,eps2", [(15, 1, 1e-4), (17, 16, 1e-4), (129, 17, 1e-4), (3000, 64, 1e-4),
                                         (3001, 200, 0.0), (2999, 3, 0.0)])
def test_groups_and_leaves(nbg, orc, gpu_ctx, solver, n, leaf, eps2):
    print(f"[walk] {solver} n={n} leaf={leaf} eps2={eps2}", flush=True)
    b = nbg.plummer(n, seed=n)
    # a third of the bodies in one place: an oversized leaf of equal keys
    for v in (b.x, b.y, b.z):
        v[: n // 3] = v[0]
    s = nbg.System(gpu_ctx, _params(nbg, solver, 0.5, leaf, eps2), n)
    s.set_state(b)
    acc = s.update_accelerations()
    counts = s.counts()
    t = orc.Tree(SOLVERS[solver], b.x, b.y, b.z, b.m, theta=0.5, leaf=leaf, bits=63, eps2=eps2)
    want, pp, npc = t.accel(b.x, b.y, b.z, counts=True)
    assert counts == (int(pp.sum()), int(npc.sum()))
    _check(acc, want)
    for k in (1, 2, 4):
        s.set_walk_split(k)
        assert np.array_equal(s.update_accelerations().view(np.uint32), acc.view(np.uint32)), f"{k} waves"
        assert s.counts() == counts
    s.close()


@pytest.mark.parametrize("solver", list(SOLVERS))
@pytest.mark.parametrize("n,theta", [(60000, 0.02), (60000, 0.1)])
def test_full_stack(nbg, orc, gpu_ctx, solver, n, theta):
    print(f"[walk] {solver} n={n} theta={theta}", flush=True)
    b = nbg.cube(n, seed=5, side=2.0)
    t = orc.Tree(SOLVERS[solver], b.x, b.y, b.z, b.m, theta=theta, leaf=1, bits=63, eps2=1e-4)
    pick = np.arange(0, n, n // 250)
    x, y, z = b.x[pick], b.y[pick], b.z[pick]
    want, pp, npc = t.accel(x, y, z, counts=True)
    s = nbg.System(gpu_ctx, _params(nbg, solver, theta, 1, 1e-4), n)
    s.set_state(b)
    got = s.accelerations_at(x, y, z)
    assert s.counts() == (int(pp.sum()), int(npc.sum()))
    s.close()
    _check(got, want)
