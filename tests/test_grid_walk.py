"""The cell-grid walk (csrc/ct_device.h, GridWalk), built for the host, against
the voxel test on every voxel: the same hits to the bit, whatever the rays do
at the lattice's planes, edges and corners.  Rays the walk does not serve (from
far away, of odd lengths, not finite) are walked through the BVH: a ray query
gets the BVH walk's hit whatever the ray."""
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


# origins up to 10^10 units away, where the grid walk's own hits differ from the
# BVH walk's at a few rays in 10^4 from about 5600 units on; a long grid,
# where the distance within it counts
@pytest.mark.parametrize("far", [30.0, 400.0, 5000.0, 2e4, 1e6, 3e9, 1e10])
@pytest.mark.parametrize("n,org", [(16, (0, 0, 0)), (12, (6000, -9000, 14000)), (0, (0, 0, 0))])
def test_queries_equal_the_bvh_walk(walk, far, n, org):
    rng = np.random.default_rng(int(far) % 1000 + n)
    if n:
        cells = np.argwhere(rng.random((n, n, n)) < 0.4) + np.array(org)
    else:
        cells = np.unique(rng.integers(0, 12, (3000, 3)) * [1, 1, 900], axis=0)
    cells, rays = np.ascontiguousarray(cells, np.int32), 20000
    lo, hi = cells.min(0) / 32.0, (cells.max(0) + 1) / 32.0
    d = rng.normal(size=(rays, 3))
    d[::5] = rng.choice([-1.0, 0.0, 1.0, 1e-6], size=(len(d[::5]), 3))
    d[np.abs(d).sum(1) == 0] = [1, 0, 0]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    to = cells[rng.integers(0, len(cells), rays)] / 32.0 + rng.uniform(0, 1 / 32.0, (rays, 3))
    o = np.ascontiguousarray(to - d * far * rng.uniform(0.5, 1.0, (rays, 1)), np.float32)
    d = np.ascontiguousarray(d * np.where(rng.random((rays, 1)) < 0.1, 10.0 ** rng.uniform(-35, 35, (rays, 1)), 1), np.float32)
    odd = slice(0, 40)
    d[odd] = rng.choice(np.array([0, -0.0, np.inf, -np.inf, np.nan, 1, 1e-42, 1e38], np.float32), size=(40, 3))
    o[20:40] = rng.choice(np.array([0, np.inf, np.nan, 0.25, 1e38], np.float32), size=(20, 3))
    for mode in (0, 1, 2):
        limit, target = np.full(rays, 1e30, np.float32), np.full(rays, NONE, np.uint32)
        limit[::11] = np.inf
        if mode == 0:
            limit[::2] = (far * rng.uniform(0.4, 1.2, len(limit[::2]))).astype(np.float32)
            target[::3] = rng.integers(0, len(cells), len(target[::3]))
        t, i, tr, ir = (np.zeros(rays, k) for k in (np.float32, np.uint32, np.float32, np.uint32))
        wide = np.zeros(rays, np.uint8)
        walk.query_and_bvh(_p(cells), len(cells), _p(IDENTITY), mode, rays, _p(o), _p(d), _p(limit), _p(target), _p(t),
                           _p(i), _p(tr), _p(ir), _p(wide))
        bad = (i != ir) | (t.view(np.uint32) != tr.view(np.uint32))
        assert not bad.any(), (mode, int(bad.sum()), o[bad][:3], d[bad][:3])
        if n == 16 and far == 30.0:  # ordinary rays stay in the grid
            assert wide[40:].mean() < 0.1
        if far >= 2e4:
            assert wide.mean() > 0.9


def _m44(rot, t):
    m = np.eye(4, dtype=np.float64)
    m[:3, :3], m[:3, 3] = rot, t
    return m


def _colmajor(m):
    return np.ascontiguousarray(m.T.reshape(16), np.float32)


def test_reach_of_transforms(walk):
    """How far from the world's origin rays may start: anywhere under the
    identity, nearer the further the instances lie, nowhere when the two
    matrices are not each other's inverses."""
    walk.reach_of.restype = C.c_float
    lo, hi = np.full(3, -4, np.float32), np.full(3, 4, np.float32)

    def reach(m, w=None):
        w = np.linalg.inv(m.astype(np.float32).astype(np.float64)) if w is None else w
        return walk.reach_of(_p(_colmajor(m)), _p(_colmajor(w)), _p(lo), _p(hi))

    rng = np.random.default_rng(3)
    q = np.linalg.qr(rng.normal(size=(3, 3)))[0]
    eye = np.eye(3)
    assert reach(_m44(eye, 0)) == np.inf
    near, far = reach(_m44(eye, [3, 0, 0])), reach(_m44(eye, [60, -20, 7]))
    assert 20 < far < near < 215
    assert 20 < reach(_m44(q, [0.1, 0, 0])) < 215
    assert 20 < reach(_m44(q * 3.0, 0)) < 215
    assert reach(_m44(eye, [500, 0, 0])) == 0.0
    assert reach(_m44(q, 0), _m44(eye, 0)) == 0.0
    assert reach(_m44(eye, 0), _m44(eye, [1e-3, 0, 0])) == 0.0
    assert reach(_m44(eye * 0.0, 0), _m44(eye * 0.0, 0)) == 0.0
    assert reach(_m44(q * 1e12, 0)) == 0.0
    p = _m44(eye, 0)
    p[3, 0] = 0.1
    assert reach(p) == 0.0
    assert reach(_m44(eye, [np.nan, 0, 0]), _m44(eye, 0)) == 0.0


def test_served_cameras_have_no_wide_ray(walk):
    """A grid that a frame keeps serves every ray from its camera and its
    scene; far and odd cameras lose it."""
    rng = np.random.default_rng(11)
    cells = np.ascontiguousarray(np.argwhere(rng.random((24, 24, 24)) < 0.2) + [-12, 5, 3000], np.int32)
    lo, hi = (cells.min(0) / 32.0).astype(np.float32), ((cells.max(0) + 1) / 32.0).astype(np.float32)
    kept = []
    for dist in (0.0, 1.0, 30.0, 80.0, 150.0, 300.0, 1e4, 1e9, np.inf, np.nan):
        for scale in (1.0, 1e-12, 1e12, 0.0, np.nan):
            rot = np.linalg.qr(rng.normal(size=(3, 3)))[0] * scale
            eye = (lo + hi) / 2 + np.array([dist, 0, 0])
            view = _colmajor(_m44(rot, eye))
            if walk.served(_p(cells), len(cells), _p(IDENTITY), C.c_float(np.inf), _p(lo), _p(hi), _p(view)):
                kept.append((dist, scale))
                n = 3000
                o = np.where(rng.random((n, 1)) < 0.5, eye, rng.uniform(lo, hi, (n, 3)))
                o, d = np.ascontiguousarray(o, np.float32), np.ascontiguousarray(rng.normal(size=(n, 3)), np.float32)
                out = [np.zeros(n, k) for k in (np.float32, np.uint32, np.float32, np.uint32, np.uint8)]
                limit, target = np.full(n, 1e9, np.float32), np.full(n, NONE, np.uint32)
                walk.query_and_bvh(_p(cells), len(cells), _p(IDENTITY), 1, n, _p(o), _p(d), _p(limit), _p(target),
                                   *(_p(x) for x in out))
                assert not out[4].any(), (dist, scale, o[out[4] > 0][:3], d[out[4] > 0][:3])
    assert {(k, 1.0) for k in (0.0, 1.0, 30.0)} <= set(kept)
    assert all(k[0] < 300 and k[1] == 1.0 for k in kept)
    view = _colmajor(_m44(np.array([[1, 1, 0], [0, 1e-6, 0], [0, 0, 1]]), (lo + hi) / 2))
    assert not walk.served(_p(cells), len(cells), _p(IDENTITY), C.c_float(np.inf), _p(lo), _p(hi), _p(view))


@pytest.mark.parametrize("count", [0, 1, 64, 65, 2097152, 2097153, 1 << 31, (1 << 32) - 2097152, (1 << 32) - 1])
def test_strided_batches_end(walk, count):
    stride = 2097152  # 64 rays for each wave of a full grid
    for base in (0, 64, stride - 64):
        want = 0 if base >= count else -(-(count - base) // stride)
        assert walk.batches(base, C.c_uint32(count), stride, 10000) == want


def test_refused_grid_memory_leaves_no_error(walk):
    """Without memory for its grid a scene is built all the same (and walked
    through its BVH); the runtime's error state must be clear for the
    launches that follow."""
    assert walk.refused_memory() == 0


def test_updates_touch_the_grid_where_the_scene_changed(walk):
    """40 instances of 64 voxels in a row: what each update does to the grid."""
    n = 40
    NONE_, KEEP, PART, FULL, ONE, GIVE_UP = 0, 1, 2, 3, 16, 32

    def plan(first=(), prims=(), shift=(), bits=(), everything=0, given_up=0):
        f, p = np.arange(n, dtype=np.uint32) * 64, np.full(n, 64, np.uint32)
        s, b = np.zeros(n, np.float32), np.ones(n, np.uint8)
        for a, edits in ((f, first), (p, prims), (s, shift), (b, bits)):
            for i, v in edits:
                a[i] = v
        lists, region = np.zeros(n, np.uint32), np.zeros(2, np.uint32)
        kind = walk.plan_update(n, _p(f), _p(p), _p(s), _p(b), everything, given_up, _p(lists), _p(region))
        return kind, {int(i): int(lists[i]) for i in np.flatnonzero(lists)}, tuple(int(v) for v in region)

    assert plan()[:2] == (KEEP | ONE, {})                                # nothing moved
    k, lists, region = plan(bits=[(20, 3)])                              # one instance: its voxels, its blocks
    assert (k, lists) == (PART | ONE, {20: 3})
    assert region[1] - region[0] <= 5 and 16 * region[0] - 16 <= 8 * 20 - 17 and 16 * region[1] - 16 >= 8 * 21 + 17
    assert plan(prims=[(7, 63)])[:2] == (PART | ONE, {7: 3})             # a voxel fewer
    assert plan(first=[(7, 9000)])[:2] == (PART | ONE, {7: 3})           # other slots
    assert plan(bits=[(7, 0)])[:2] == (PART | ONE, {7: 1})               # an instance gone
    assert plan(bits=[(7, 3), (9, 5)])[:2] == (PART | ONE, {7: 3, 9: 4})  # a bad one is tried again
    assert plan(bits=[(9, 5)])[:2] == (KEEP | ONE, {})                   # but not when nothing made room
    assert plan(bits=[(i, 5) for i in range(6)] + [(20, 3)])[0] == NONE_ | ONE | GIVE_UP
    assert plan(bits=[(20, 3)], given_up=1)[0] == NONE_ | ONE | GIVE_UP
    assert plan(given_up=1, everything=1)[0] == FULL | ONE
    assert plan(shift=[(39, 200.0)], bits=[(39, 3)])[0] == FULL | ONE    # out of the grid
    assert plan(bits=[(i, 3) for i in range(21)])[0] == FULL | ONE       # more than half of it
    assert plan(bits=[(i, 3) for i in range(20)])[0] == PART | ONE
    assert plan(everything=1)[0] == FULL | ONE
    assert plan(bits=[(5, 9)])[:2] == (KEEP, {})                         # moved by its transform: the arrays stay right
    assert plan(bits=[(5, 9), (6, 3)])[0] == NONE_
    assert plan(shift=[(3, 1e9)], bits=[(3, 3)])[0] == NONE_ | ONE       # out of range
    assert plan(shift=[(3, np.nan)], bits=[(3, 3)])[0] in (NONE_ | ONE, FULL | ONE)
    assert plan(bits=[(i, 0) for i in range(n)])[0] == NONE_             # an empty scene
