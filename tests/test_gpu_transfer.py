"""Host copies of state arrays through pinned slots: every size at which the
path changes (words left over, one slot or many, one thread or four, uploads
that fit a slot or not) gives back what was put in, the interleaved
accelerations are the separate ones, and threads that share a context do not
meet in the slots."""

import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz")


def _bodies(nbg, n, seed):
    r = np.random.default_rng(seed)
    return nbg.Bodies(*(r.uniform(-1, 1, n).astype(np.float32) for _ in range(7)))


def _separate(nbg, s, n):
    a = [np.zeros(n, np.float32) for _ in range(3)]
    ptr = [v.ctypes.data_as(ctypes.POINTER(ctypes.c_float)) for v in a]
    assert nbg.lib().nbg_sys_get_accelerations(s.handle, *ptr) == 0
    return np.stack(a, 1)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 37448, 37449, 43688, 43689, 87381, 349504, 349529, 700001])
def test_roundtrip(nbg, gpu_ctx, n):
    b = _bodies(nbg, n, n)
    p = nbg.default_params()
    p.solver, p.theta, p.sum_mode = nbg.BARNES_HUT, 1.5, nbg.SUM_FAST
    s = nbg.System(gpu_ctx, p, n)
    s.set_state(b)
    got = s.get_state()
    for f in FIELDS:
        assert np.array_equal(getattr(got, f), getattr(b, f)), f
    a = s.update_accelerations()
    assert a.shape == (n, 3) and a.flags.c_contiguous
    assert np.array_equal(a.view(np.uint32), _separate(nbg, s, n).view(np.uint32))
    s.close()


def test_members_and_threads(nbg, gpu_ctx):
    p = nbg.default_params()
    p.solver, p.theta, p.morton_bits = nbg.LINEAR_BVH, 1.0, 30
    bad = []

    def work(k):
        sizes = [1, 30 + k, 4099, 90001]
        sets = [_bodies(nbg, n, 10 * k + i) for i, n in enumerate(sizes)]
        batch = nbg.Batch(gpu_ctx, sum(sizes), 8)
        ids = [batch.add(p, b) for b in sets]
        batch.update_accelerations()
        for i, b in zip(ids, sets):
            st, acc = batch.get(i, accelerations=True)
            if not all(np.array_equal(getattr(st, f), getattr(b, f)) for f in FIELDS):
                bad.append((k, b.n, "state"))
            s = nbg.System(gpu_ctx, p, b.n)
            s.set_state(b)
            q = nbg.default_params()
            q.solver, q.theta, q.morton_bits, q.sum_mode = p.solver, p.theta, p.morton_bits, nbg.SUM_FAST
            s.params = q
            if not np.array_equal(s.update_accelerations().view(np.uint32), acc.view(np.uint32)):
                bad.append((k, b.n, "accelerations"))
            s.close()
        batch.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
