"""Kernels run on the CPU, a workgroup's threads as fibres that go on until
they need one another (tests/native/simt.hpp): a wave gets as far ahead of the
others as the barriers let it, whatever the order of the waves, and
AddressSanitizer sees every access.  For races and reads out of bounds, which
no GPU run would show."""

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "n-body_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")


def _clang():
    for c in ("/opt/rocm/lib/llvm/bin/clang++", "/opt/rocm/llvm/bin/clang++", shutil.which("clang++")):
        if c and os.path.exists(c):
            return c
    return None


pytestmark = pytest.mark.skipif(_clang() is None, reason="needs clang++")


def _build(out, check, kernels, asan):
    """The check program with the kernel files it needs, built in parallel."""
    flags = [_clang(), "-std=c++17", "-O0", "-gline-tables-only", "-w", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
             "-I/opt/rocm/include", "-I" + CSRC]
    if asan:
        flags += ["-fsanitize=address", "-fno-omit-frame-pointer", "-DSIMT_REDZONES"]
    jobs, objs = [], []
    for src in [os.path.join(CSRC, k + ".hip") for k in kernels] + [os.path.join(NATIVE, f) for f in ("simt.cpp", check)]:
        obj = os.path.join(out, os.path.basename(src) + ".o")
        shim = ["-include", os.path.join(NATIVE, "simt.hpp")] if src.endswith(".hip") else []
        jobs.append(subprocess.Popen([*flags, *shim, "-x", "c++", "-c", src, "-o", obj], stderr=subprocess.PIPE))
        objs.append(obj)
    for j in jobs:
        err = j.communicate()[1]
        assert j.returncode == 0, err.decode()[-4000:]
    exe = os.path.join(out, "check")
    subprocess.run([*flags, *objs, "-o", exe], check=True)
    return exe


def _run(exe, *args, order=0):
    env = dict(os.environ, NBG_SIMT_ORDER=str(order), ASAN_OPTIONS="detect_leaks=0:detect_stack_use_after_return=0")
    return subprocess.run([exe, *args], capture_output=True, text=True, timeout=600, env=env)


def test_target_groups(tmp_path):
    exe = _build(str(tmp_path), "targets_check.cpp", ["targets"], asan=False)
    outs = []
    for order in (0, 1, 2, 3):
        r = _run(exe, order=order)
        assert r.returncode == 0, f"order {order}\n" + r.stdout[-2000:] + r.stderr[-2000:]
        outs.append(r.stdout)
    assert len(set(outs)) == 1


def test_frames_without_a_root(tmp_path):
    exe = _build(str(tmp_path), "frames_check.cpp", ["walk", "walk_fast"], asan=True)
    r = _run(exe)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("what", ["failed", "runs", "fills"])
def test_last_stage_of_the_sort(tmp_path, what):
    exe = _build(str(tmp_path), "sort_check.cpp", ["build"], asan=True)
    r = _run(exe, what)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


# n, leaf, max_depth, coincident bodies
@pytest.mark.parametrize("n,leaf,depth,same", [(3000, 2, 12, 129), (700, 1, 32, 65), (1500, 64, 5, 700)])
def test_octree_pass_in_bounds(octree_exe, tmp_path, nbg, orc, n, leaf, depth, same):
    """Box to ORDERED walk with buffers exactly as large as the library makes
    them: no access outside them, and the oracle's bits."""
    b = nbg.plummer(n, seed=300 + n)
    for a in (b.x, b.y, b.z):
        a[n // 3:n // 3 + same] = a[n // 3]
    np.concatenate([b.x, b.y, b.z, b.m]).tofile(tmp_path / "in")
    r = _run(octree_exe, str(tmp_path / "in"), str(n), str(leaf), str(depth), "0.9", "1e-4", str(tmp_path / "out"), "0",
             str(n), "1")
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    acc = np.fromfile(tmp_path / "out", np.float32).reshape(n, 3)
    t = orc.Tree(0, b.x, b.y, b.z, b.m, theta=0.9, leaf=leaf, max_depth=depth, eps2=1e-4)
    assert np.array_equal(acc.view(np.uint32), np.asarray(t.accel(b.x, b.y, b.z)).view(np.uint32))


@pytest.mark.parametrize("n,leaf,same", [(700, 16, 65), (500, 130, 0)])
def test_fast_walk_in_bounds(octree_exe, tmp_path, nbg, orc, n, leaf, same):
    """The FAST walk's lists, queues and stack, the waves in a shuffled order:
    no access out of bounds, and the oracle's interaction counts."""
    b = nbg.plummer(n, seed=300 + n)
    for a in (b.x, b.y, b.z):
        a[n // 3:n // 3 + same] = a[n // 3]
    np.concatenate([b.x, b.y, b.z, b.m]).tofile(tmp_path / "in")
    r = _run(octree_exe, str(tmp_path / "in"), str(n), str(leaf), "20", "0.5", "1e-4", str(tmp_path / "out"), "0", str(n),
             "0", order=3)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    t = orc.Tree(0, b.x, b.y, b.z, b.m, theta=0.5, leaf=leaf, max_depth=20, eps2=1e-4)
    _, pp, npc = t.accel(b.x, b.y, b.z, counts=True)
    assert f"pp {int(pp.sum())} np {int(npc.sum())}" in r.stdout


@pytest.fixture(scope="module")
def octree_exe(tmp_path_factory):
    return _build(str(tmp_path_factory.mktemp("octree")), "octree_check.cpp", ["build", "octree", "walk", "walk_fast"],
                  asan=True)


def test_forest_order_of_workgroups(tmp_path):
    """Members of 16,384 bodies are eight runs of 32 workgroups each: with run x
    of eight always on XCD x, every member's dense eighth was on one XCD."""
    exe = _build(str(tmp_path), "turns_check.cpp", [], False)
    rows = [r.split() for r in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(rows) == 40
    # most of one eighth of all members that is on one XCD, 1: shared evenly, 8: all of it
    uneven = [r for r in rows if int(r[0]) >= 64 and float(r[2]) > 1.3]
    assert not uneven, uneven
