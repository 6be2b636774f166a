"""The cell-grid walk (csrc/ct_device.h, GridWalk), built for the host, against
the voxel test on every voxel: the same hits to the bit, whatever the rays do
at the lattice's planes, edges and corners."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and os.path.exists(c)), None)
NONE = 0xFFFFFFFF
IDENTITY = np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], np.float32)


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    if CLANG is None:
        pytest.skip("no clang++ (the device header uses its vector types)")
    out = str(tmp_path_factory.mktemp("walk") / "libwalk.so")
    src = os.path.join(HERE, "host_walk")
    subprocess.run([CLANG, "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-fopenmp", "-I", src, "-o", out,
                    os.path.join(src, "walk_host.cpp")], check=True)
    return C.CDLL(out)


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _both(lib, cells, w2o, mode, o, d, limit, target):
    n = len(o)
    t, i, tr, ir = np.zeros(n, np.float32), np.zeros(n, np.uint32), np.zeros(n, np.float32), np.zeros(n, np.uint32)
    lib.walk_and_brute(_p(cells), len(cells), _p(w2o), mode, n, _p(o), _p(d), _p(limit), _p(target), _p(t), _p(i), _p(tr),
                       _p(ir))
    return (i != ir) | (t.view(np.uint32) != tr.view(np.uint32)), ir


def _rays(rng, n, cells, kind):
    lo, hi = cells.min(0) / 32.0, (cells.max(0) + 1) / 32.0
    ext = (hi - lo).max()
    d = rng.normal(size=(n, 3))
    if kind == "axis":  # along an axis, or so nearly that it is crossed once or never
        d *= np.where(rng.random((n, 3)) < 0.5, rng.choice([0, 0, 1e-12, 1e-7, 1e-5, 1e-3], size=(n, 3)), 1)
        d[np.abs(d).sum(1) == 0] = [1, 0, 0]
    elif kind == "diagonal":  # two and three planes crossed at once
        d = rng.choice([-1, 0, 1, 0.5], size=(n, 3)).astype(float)
        d[np.abs(d).sum(1) == 0] = [1, 1, 1]
    if kind == "scaled":
        d *= 10.0 ** rng.uniform(-6, 6, (n, 1))
    else:
        d /= np.linalg.norm(d, axis=1, keepdims=True)
    to = rng.uniform(lo, hi, (n, 3))
    if kind in ("axis", "diagonal", "edge"):  # through lattice points, edges, faces and centres, or just beside them
        q = np.round(to * 32) / 32
        to = np.where(rng.random((n, 3)) < 0.6, q, np.where(rng.random((n, 3)) < 0.5, q + 1 / 64.0, to))
        to = to + np.where(rng.random((n, 3)) < 0.3, rng.choice([1e-7, -1e-7, 1e-6, -1e-5, 1.5e-5], size=(n, 3)), 0)
    un = d / np.linalg.norm(d, axis=1, keepdims=True)
    o = to - un * rng.choice([0, 0, 0.1, 1.0, 3.0, 20.0], size=(n, 1)) * ext
    return np.ascontiguousarray(o, np.float32), np.ascontiguousarray(d, np.float32)


def _rotation(rng):
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return np.concatenate([q.T.reshape(9), rng.normal(size=3) * 0.1]).astype(np.float32)


# one voxel; a brick's corner and far from the origin; solid; bricks and cubes
# of bricks that are empty; two voxels in opposite corners
@pytest.mark.parametrize("n,fill,org", [(1, 1.0, (0, 0, 0)), (5, 0.5, (-3, 7, 100)), (16, 0.9, (1000, -2000, 31)),
                                        (20, 0.05, (-30, 5, -17)), (40, 0.0006, (-20, -20, -20)),
                                        (90, 0.00008, (-45, 3, 11)), (70, 0.0, (0, 0, -70))])
@pytest.mark.parametrize("kind", ["random", "axis", "diagonal", "edge", "scaled"])
def test_walk_equals_every_voxel(walk, n, fill, org, kind):
    rng = np.random.default_rng(n * 7 + len(kind))
    cells = np.argwhere(rng.random((n, n, n)) < fill)
    if fill == 0.0:
        cells = np.array([[0, 0, 0], [n - 1] * 3])
    cells = np.ascontiguousarray(cells + np.array(org), np.int32)
    rays, hits = 4000, 0
    for w2o in (IDENTITY, _rotation(rng)):
        o, d = _rays(rng, rays, cells, kind)
        if w2o is not IDENTITY:  # aim in world space: o' = R^T (o - b)
            m = w2o[:9].reshape(3, 3).T.astype(np.float64)
            o = np.ascontiguousarray((o - w2o[9:].astype(np.float64)) @ m, np.float32)
            d = np.ascontiguousarray(d @ m, np.float32)
        for mode in (0, 1, 2):  # any hit, closest, path segment
            limit, target = np.full(rays, 1e9, np.float32), np.full(rays, NONE, np.uint32)
            if mode == 0:
                limit = (rng.uniform(0, 1, rays) * n / 32 * 3 / np.linalg.norm(d, axis=1)).astype(np.float32)
                limit[::7], limit[::50] = 1e9, 0.0
                target[::2] = rng.integers(0, len(cells), rays // 2)
            bad, ref = _both(walk, cells, w2o, mode, o, d, limit, target)
            assert not bad.any(), (mode, o[bad][:3], d[bad][:3])
            hits += int((ref == 1).sum() if mode == 0 else (ref != NONE).sum())
    assert hits or fill < 0.001


def test_rays_that_hit_nothing(walk):
    """Zero, infinite and NaN directions and origins end at once, as misses."""
    cells = np.ascontiguousarray(np.argwhere(np.ones((6, 6, 6))), np.int32)
    bad_values = [(0, 0, 0), (np.inf, 0, 0), (np.nan, 1, 0), (0, -np.inf, np.inf), (0.0, -0.0, 0.0)]
    o = np.array([(0.1, 0.1, 0.1)] * 5 + [(np.nan, 0.1, 0.1), (np.inf, 0.1, 0.1), (0.1, -np.inf, 0.1)], np.float32)
    d = np.array(bad_values + [(0, 0, 1)] * 3, np.float32)
    limit, target = np.full(len(o), 1e9, np.float32), np.full(len(o), NONE, np.uint32)
    for mode in (0, 1, 2):
        bad, ref = _both(walk, cells, IDENTITY, mode, o, d, limit, target)
        assert not bad.any()
        assert (ref == (0 if mode == 0 else NONE)).all()
