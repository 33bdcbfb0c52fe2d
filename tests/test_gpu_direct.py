"""FAST direct sum at the sizes where its split of the sources over a
workgroup's waves can go wrong: fewer sources than waves, shares of less than
four sources, shares that end inside a run, and the last share empty."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps2", [1e-4, 0.0])
@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 961, 1023, 1025, 4100, 16385])
def test_fast_direct_matches_oracle(nbg, orc, gpu_ctx, n, eps2):
    print(f"[direct] n={n} eps2={eps2}", flush=True)
    b = nbg.cube(n, seed=7 + n, side=2.0)
    p = nbg.default_params()
    p.solver, p.eps2, p.sum_mode = nbg.NAIVE, eps2, nbg.SUM_FAST
    s = nbg.System(gpu_ctx, p, n)
    s.set_state(b)
    acc = s.update_accelerations()
    assert s.counts() == (n * n, 0)
    pts = np.random.default_rng(n).uniform(-1, 1, (70, 3)).astype(np.float32)
    at = s.accelerations_at(pts[:, 0], pts[:, 1], pts[:, 2])
    s.close()
    for got, x, y, z in ((acc, b.x, b.y, b.z), (at, *pts.T.copy())):
        ref = orc.direct_f32(b.x, b.y, b.z, b.m, x, y, z, 1.0, eps2)
        mag = np.linalg.norm(ref, axis=1)
        floor = max(float(np.sqrt(np.mean(mag ** 2))), 1e-30)
        # the FAST bound of every solver: FP32 sums of up to 64 terms, rsqrt within an ulp
        assert np.max(np.linalg.norm(got - ref, axis=1) / np.maximum(mag, floor)) <= 1e-5
