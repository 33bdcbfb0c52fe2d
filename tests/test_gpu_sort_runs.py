"""The build's sort where many keys share their leading bits: bodies in
clusters far smaller than the box (one long run, many, more than the run list
holds), coincident bodies, and sizes at the edges of its tiles.  Keys and
permutation are the oracle's stable order; the octree, whose cells depend on
the second key word there, gives the oracle's bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(nbg, kind, n):
    r = np.random.default_rng(n)
    b = nbg.cube(n, seed=n, side=2.0)
    if kind == "cluster":  # everything but two bodies within 1e-6
        p = (0.25 + 1e-6 * r.uniform(-1, 1, (3, n))).astype(np.float32)
    elif kind == "coincident":
        p = np.full((3, n), 0.25, np.float32)
    elif kind == "clusters":  # groups of 260 bodies within 1e-5 of each other
        c = np.repeat(r.uniform(-1, 1, (3, n // 260 + 1)), 260, axis=1)[:, :n]
        p = (c + 1e-5 * r.uniform(-1, 1, (3, n))).astype(np.float32)
        p = p[:, r.permutation(n)]
    elif kind == "escapers":  # two bodies ten thousand sides out
        p = np.stack([b.x, b.y, b.z])
        p[:, 0], p[:, -1] = -10000.0, 10000.0
        b.x, b.y, b.z = (np.ascontiguousarray(v) for v in p)
        return b
    else:
        return b
    p[:, :1], p[:, -1:] = -1.0, 1.0
    b.x, b.y, b.z = (np.ascontiguousarray(v) for v in p)
    return b


def _params(nbg, solver, bits, leaf=16):
    p = nbg.default_params()
    p.solver, p.theta, p.leaf_size, p.morton_bits, p.eps2 = solver, 0.7, leaf, bits, 1e-4
    p.sum_mode = nbg.SUM_FAST
    return p


@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("kind,n", [("cube", 1), ("cube", 2), ("cube", 1023), ("cube", 1025), ("cube", 262145),
                                    ("cluster", 258), ("cluster", 5000), ("cluster", 40000), ("coincident", 3000),
                                    ("clusters", 5001), ("clusters", 90000), ("clusters", 1200000)])
def test_linear_bvh_order(nbg, orc, gpu_ctx, kind, n, bits):
    print(f"[sort] {kind} n={n} bits={bits}", flush=True)
    b = _bodies(nbg, kind, n)
    s = nbg.System(gpu_ctx, _params(nbg, nbg.LINEAR_BVH, bits, leaf=64), n)
    s.set_state(b)
    s.enable_counts(False)
    s.update_accelerations()
    keys, perm = s.debug_order()
    s.close()
    want = np.asarray(orc.morton(b.x, b.y, b.z, bits, orc.bbox(b.x, b.y, b.z)), np.uint64)
    order = np.argsort(want, kind="stable")
    assert np.array_equal(perm, order.astype(np.uint32))
    assert np.array_equal(keys, want[order])


@pytest.mark.parametrize("kind,n,leaf", [("cluster", 300, 1), ("cluster", 6000, 16), ("coincident", 700, 4),
                                         ("clusters", 9000, 8), ("cube", 257, 1)])
def test_octree_bits(nbg, orc, gpu_ctx, kind, n, leaf):
    print(f"[sort] octree {kind} n={n} leaf={leaf}", flush=True)
    b = _bodies(nbg, kind, n)
    p = _params(nbg, nbg.BARNES_HUT, 63, leaf=leaf)
    p.sum_mode = nbg.SUM_ORDERED
    s = nbg.System(gpu_ctx, p, n)
    s.set_state(b)
    acc = s.update_accelerations()
    t = orc.Tree(0, b.x, b.y, b.z, b.m, theta=0.7, leaf=leaf, bits=63, eps2=1e-4)
    want, pp, npc = t.accel(b.x, b.y, b.z, counts=True)
    assert np.array_equal(acc.view(np.uint32), want.view(np.uint32))
    assert s.counts() == (int(pp.sum()), int(npc.sum()))
    s.close()


@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("kind,n", [("cube", 131073), ("cube", 4194305), ("cluster", 16386), ("cluster", 16387),
                                    ("cluster", 300001), ("escapers", 1200000), ("coincident", 70000)])
def test_long_runs_order(nbg, orc, gpu_ctx, kind, n, bits):
    test_linear_bvh_order(nbg, orc, gpu_ctx, kind, n, bits)


@pytest.mark.parametrize("kind,n,leaf", [("cluster", 20000, 16), ("escapers", 150000, 8)])
def test_long_runs_octree(nbg, orc, gpu_ctx, kind, n, leaf):
    test_octree_bits(nbg, orc, gpu_ctx, kind, n, leaf)


@pytest.mark.parametrize("solver", ["LINEAR_BVH", "BARNES_HUT"])
@pytest.mark.parametrize("n", [100000, 1000000])
def test_escapers_cost(nbg, gpu_ctx, solver, n):
    """Two bodies far out put all others into a few runs.  The sort then takes
    twice the passes or three times: at 1,000,000 bodies 5 (linear BVH) and 7
    (octree) times the plain sort.  One workgroup with such a run took 26 and
    34 times."""
    ms = {}
    for kind in ("cube", "escapers"):
        b = _bodies(nbg, kind, n)
        p = _params(nbg, getattr(nbg, solver), 63)
        p.theta = 1.0
        s = nbg.System(gpu_ctx, p, n)
        s.set_state(b)
        s.enable_counts(False)
        s.enable_timing(True)
        times = []
        for _ in range(5):
            s.update_accelerations()
            times.append(s.phase_times()["sort"])
        ms[kind] = min(times)
        s.close()
    print(f"[sort] {solver} n={n} ms {ms}", flush=True)
    assert ms["escapers"] <= 12 * ms["cube"]


def test_keys_of_large_systems(nbg, gpu_ctx):
    """The keys of 16,777,216 bodies take 5 times as long as those of 1,048,576;
    with 256 workgroups of 256 threads for both it was 12 times."""
    ms = {}
    for n in (1 << 20, 1 << 24):
        p = _params(nbg, nbg.LINEAR_BVH, 63, leaf=32)
        p.theta = 1.2
        s = nbg.System(gpu_ctx, p, n)
        s.set_state(nbg.cube(n, seed=3, side=2.0))
        s.enable_counts(False)
        s.enable_timing(True)
        times = []
        for _ in range(10):
            s.update_accelerations()
            times.append(s.phase_times()["keys"])
        s.close()
        ms[n] = min(times)
    print(f"[sort] keys, ms {ms}", flush=True)
    assert ms[1 << 24] <= 8 * ms[1 << 20]
