"""Scenes with a cell grid are walked through it, except by counted launches
(`stats`), which walk the BVH: both must give the same hits to the bit, and a
scene that an update takes off the lattice must leave the grid."""
import ctypes as C

import numpy as np
import pytest

import ctamd
import oracle as O
from ctamd import adjoint as adj

pytestmark = pytest.mark.gpu


def _load(grid, chunk, fill=0.2, seed=5):
    d = ctamd.SceneDesc()
    d.grid[:] = [grid] * 3
    d.chunk[:] = [chunk] * 3
    d.occupied_count = max(1, round(fill * grid ** 3))
    d.le_min = d.le_max = 1.0
    d.albedo_min, d.albedo_max = 0.2, 0.8
    d.seed = seed
    d.voxel_extent = ctamd.CT_VOXEL_EXTENT
    sc = ctamd.Scene(d)
    acc = ctamd.Accel(max_instances=sc.info.instance_count + 8,
                      max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024, max_cube_lights=8)
    adj._load_geometry(sc, acc)
    return sc, acc


def _rays(rng, n, lo, hi):
    """Rays from around and within, a third of them through lattice planes, edges and corners or along the axes."""
    ext = float((hi - lo).max())
    d = rng.normal(size=(n, 3))
    d[::6] = rng.choice([-1.0, 0.0, 1.0], size=(len(d[::6]), 3))
    d[1::6] *= rng.choice([0.0, 1e-7, 1e-4, 1.0], size=(len(d[1::6]), 3))
    d[np.abs(d).sum(1) == 0] = [0, 1, 0]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    to = rng.uniform(lo, hi, (n, 3))
    to[::3] = np.round(to[::3] * 32) / 32 + rng.choice([0, 0, 1e-6, -1e-6, 1 / 64], size=(len(to[::3]), 3))
    o = to - d * rng.choice([0, 0.05, 1.0, 3.0], size=(n, 1)) * ext
    return np.ascontiguousarray(o, np.float32), np.ascontiguousarray(d, np.float32)


def _same(acc, sc, seed, n=60000):
    rng = np.random.default_rng(seed)
    o, d = _rays(rng, n, sc.grid_min.astype(np.float64), sc.grid_max.astype(np.float64))
    t, ids = acc.trace_closest(o, d)
    bt, bids, _ = acc.trace_closest(o, d, stats=True)
    assert np.array_equal(ids, bids) and np.array_equal(t.view(np.uint32), bt.view(np.uint32))
    assert 0.02 < (ids[:, 0] != ctamd.CT_INVALID_INDEX).mean() < 1.0
    g, b = acc.trace_bounce(o, d), acc.trace_bounce(o, d, stats=True)
    for k in ("ids", "pos", "nrm", "dist", "wo"):
        assert np.array_equal(g[k].view(np.uint32), b[k].view(np.uint32)), k
    hit = ids[:, 0] != ctamd.CT_INVALID_INDEX
    dist = np.where(hit, t * rng.choice([0.5, 1.0, 1.5], size=n), 2.0).astype(np.float32)
    targets = np.where((rng.random(n) < 0.5)[:, None], ids, ctamd.CT_INVALID_INDEX).astype(np.uint32)
    for tg in (None, targets):
        occ, (bocc, _) = acc.trace_any(o, d, dist, tg), acc.trace_any(o, d, dist, tg, stats=True)
        assert np.array_equal(occ, bocc)


@pytest.mark.parametrize("grid,chunk,fill", [(1, 1, 1.0), (3, 3, 0.5), (17, 5, 0.3), (64, 16, 0.2), (130, 64, 0.02)])
def test_grid_walk_equals_bvh_walk(gpu, grid, chunk, fill):
    sc, acc = _load(grid, chunk, fill)
    _same(acc, sc, grid)


def test_grid_follows_updates(gpu):
    sc, acc = _load(48, 16)
    _same(acc, sc, 1)
    n = [i.primitive_count for i in acc.read_instances()]
    big = int(np.argmax(n))
    box = acc.read_world()["aabbs"]
    first = [i.first_primitive_index for i in acc.read_instances()]
    old = box[first[big]].copy()
    acc.delete_primitive(big, 3)  # the voxel leaves the grid
    acc.update_scene()
    _same(acc, sc, 2)
    acc.undo()
    acc.update_scene()
    _same(acc, sc, 3)
    acc.update_blas(big, edits=[(0, old + np.float32(0.007))])  # off the lattice
    acc.update_scene()
    _same(acc, sc, 4)
    acc.update_blas(big, edits=[(0, box[first[big] + 1])])  # two voxels in one cell
    acc.update_scene()
    _same(acc, sc, 5)
    acc.update_blas(big, edits=[(0, old + np.float32(0.5))])  # another cell of the lattice
    acc.update_scene()
    _same(acc, sc, 6)
    acc.update_blas(big, edits=[(0, old)])
    acc.update_scene()
    m = np.eye(4, dtype=np.float32)
    m[3, 0] = 0.25
    acc.update_blas(big, transform=m.reshape(16))  # instances with different transforms
    acc.update_scene()
    _same(acc, sc, 7)
    m[3, 0] = -0.25
    acc.update_blas(big, transform=m.reshape(16))
    acc.update_scene()
    _same(acc, sc, 8)


def test_grid_under_one_transform(gpu):
    """A scene placed by one rotation and translation keeps its grid."""
    d = ctamd.hd_di(width=16, height=16, grid=48, chunk=16)
    sc = ctamd.Scene(ctamd.scene_desc(d))
    acc = ctamd.Accel(max_instances=sc.info.instance_count + 8,
                      max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024,
                      max_cube_lights=sc.info.cube_light_count + 8)
    ctx = ctamd.Ctx(16, 16)
    c, s = np.cos(0.7), np.sin(0.7)
    m = np.array([[c, 0, -s, 0], [0, 1, 0, 0], [s, 0, c, 0], [0.1, -0.2, 0.05, 1]], np.float32)
    ctamd.load_scene(sc, acc, ctx, transform=m.reshape(16))
    _same(acc, sc, 9)


def test_far_rays_take_the_bvh(gpu):
    """Rays from up to 10^10 units away, of odd lengths and not finite: the
    counted walk's hits, to the bit (the grid's own differ from about 5600
    units on)."""
    sc, acc = _load(16, 16, 0.4)
    rng = np.random.default_rng(4)
    n = 200000
    lo, hi = sc.grid_min.astype(np.float64), sc.grid_max.astype(np.float64)
    for far in (300.0, 2e4, 1e6, 3e9):
        d = rng.normal(size=(n, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        o = np.ascontiguousarray(rng.uniform(lo, hi, (n, 3)) - d * far, np.float32)
        d = np.ascontiguousarray(d * np.where(rng.random((n, 1)) < 0.1, 10.0 ** rng.uniform(-30, 30, (n, 1)), 1), np.float32)
        d[:40] = rng.choice(np.array([0, -0.0, np.inf, np.nan, 1, 1e-42, 1e38], np.float32), size=(40, 3))
        o[20:40] = rng.choice(np.array([0, np.inf, np.nan, 0.25, 1e38], np.float32), size=(20, 3))
        t, ids = acc.trace_closest(o, d, tmax=1e30)
        bt, bids, _ = acc.trace_closest(o, d, tmax=1e30, stats=True)
        assert np.array_equal(ids, bids) and np.array_equal(t.view(np.uint32), bt.view(np.uint32))
        g, b = acc.trace_bounce(o, d), acc.trace_bounce(o, d, stats=True)
        for k in ("ids", "pos", "nrm", "dist", "wo"):
            assert np.array_equal(g[k].view(np.uint32), b[k].view(np.uint32)), k
        dist = np.full(n, np.float32(far * 1.5))
        occ, (bocc, _) = acc.trace_any(o, d, dist, ids), acc.trace_any(o, d, dist, ids, stats=True)
        assert np.array_equal(occ, bocc)


@pytest.mark.parametrize("far", [12.0, 2e4, 1e5])
def test_frames_of_far_cameras(gpu, far):
    """Frames from a camera far outside the scene: the bits of frames that walk
    the BVH (instrumented ones)."""
    w = ctamd.hd_di(width=640, height=360, grid=32, chunk=16)
    scenes = [ctamd.Scene(ctamd.scene_desc(w)) for _ in range(2)]
    lo, hi = scenes[0].grid_min.astype(np.float64), scenes[0].grid_max.astype(np.float64)
    back = np.array([0.48, 0.6, 0.64])
    eye = (lo + hi) / 2 + far * back
    # the library's camera loses the direction in the position's rounding
    right = np.cross([0.0, 1.0, 0.0], back)
    right /= np.linalg.norm(right)
    view = np.zeros((4, 4))
    view[:3, 0], view[:3, 1], view[:3, 2], view[:3, 3], view[3, 3] = right, np.cross(back, right), back, eye, 1.0
    w.fov_radians = 1.2 * float((hi - lo).max()) / far

    def params(f):
        p = ctamd.frame_params(w, f)
        p.inv_view[:] = np.float32(view.T.reshape(16)).tolist()
        return p

    images = []
    for k in range(2):
        sc = scenes[k]
        acc = ctamd.Accel(max_instances=sc.info.instance_count + 8,
                          max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024,
                          max_cube_lights=sc.info.cube_light_count + 8)
        ctx = ctamd.Ctx(w.width, w.height)
        ctamd.load_scene(sc, acc, ctx)
        ctx.set_instrumentation(2 if k else 0)
        for f in range(2):
            ctx.render(acc, params(f))
        images.append((ctx.read(ctamd.CT_BUF_IMAGE, w.width, w.height), bytes(ctx.read(ctamd.CT_BUF_DI, w.width, w.height))))
    hits = (np.frombuffer(images[1][1], np.float32).reshape(-1, 15)[:, 3] > 0).mean()
    assert 0.1 < hits < 1.0, hits
    assert np.array_equal(images[0][0].view(np.uint32), images[1][0].view(np.uint32))
    assert images[0][1] == images[1][1]


def _add_instance(acc, boxes, prims):
    """A BUILD task of one instance."""
    st = acc.staging()
    st.instances[0].first_primitive_index = 0
    st.instances[0].primitive_count = len(boxes)
    b, p = np.ascontiguousarray(boxes, np.float32), np.ascontiguousarray(prims, np.uint32)
    C.memmove(st.aabbs, b.ctypes.data, b.nbytes)
    C.memmove(st.primitives, p.ctypes.data, p.nbytes)
    t = ctamd.Task()
    t.type = ctamd.CT_TASK_BUILD_BLAS_FROM_CPU
    t.u.blas_build_from_cpu.instance_count = 1
    t.u.blas_build_from_cpu.primitive_count = len(boxes)
    for k in range(16):
        t.u.blas_build_from_cpu.transform[k] = 1.0 if k % 5 == 0 else 0.0
    acc.task_queue_add(t)


# instances that share bricks (chunks of 5 and 6 cells), a brick's multiple, one
# instance; the sequences take the grid away and bring it back
@pytest.mark.parametrize("grid,chunk,fill", [(17, 5, 0.3), (24, 6, 0.6), (48, 16, 0.1), (90, 30, 0.01), (12, 12, 0.5)])
def test_grid_follows_edit_sequences(gpu, grid, chunk, fill):
    sc, acc = _load(grid, chunk, fill, seed=grid)
    rng = np.random.default_rng(grid)
    step = np.eye(4, dtype=np.float32)
    back, at = [], 0
    cell = np.float32(1 / 32)

    def update():
        nonlocal at
        acc.update_scene()
        at += 1
        print("edit", grid, at, flush=True)
        _same(acc, sc, 100 + at, n=12000)

    for _ in range(24):
        while back:
            back.pop()()
            update()
        insts = acc.read_instances()
        used = [i for i, r in enumerate(insts) if r.primitive_count > 4]
        inst = int(rng.choice(used))
        r, box = insts[inst], acc.read_world()["aabbs"]
        first, n = r.first_primitive_index, r.primitive_count
        op = rng.choice(["delete", "two", "brush", "move", "off", "double", "shift", "drop", "still", "grow"])
        if op == "delete":
            acc.delete_primitive(inst, int(rng.integers(0, n)))
            if rng.random() < 0.5:
                back.append(acc.undo)
        elif op == "two":  # two instances in one update
            other = int(rng.choice(used))
            acc.delete_primitive(inst, 0)
            acc.delete_primitive(other, 1)
        elif op == "brush":
            acc.brush_mark([(inst, int(p)) for p in rng.choice(n, 2, replace=False)])
            acc.process_voxel_modifications()
        elif op in ("move", "off", "double", "grow"):
            p = int(rng.integers(0, n))
            old = box[first + p].copy()
            other = insts[int(rng.choice(used))].first_primitive_index
            new = {"move": old + cell * np.tile(rng.integers(-3, 4, 3), 2), "off": old + np.float32(0.007),
                   "double": box[other].copy(), "grow": old + np.float32(0.5 * (1 + at % 3))}[op]
            acc.update_blas(inst, edits=[(p, new.astype(np.float32))])
            back.append(lambda i=inst, p=p, b=old: acc.update_blas(i, edits=[(p, b)]))
        elif op == "shift":
            m = step.copy()
            m[3, 0] = 0.25
            acc.update_blas(inst, transform=m.reshape(16))
            m = m.copy()
            m[3, 0] = -0.25
            back.append(lambda i=inst, m=m: acc.update_blas(i, transform=m.reshape(16)))
        elif op == "drop" and len(used) > 1:
            boxes, prims = box[first:first + n].copy(), acc.read_world()["prims"][first:first + n].copy()
            acc.delete_blas(inst)
            back.append(lambda b=boxes, p=prims: _add_instance(acc, b, p))
        else:
            acc.update_blas(inst, transform=step.reshape(16))
        update()


def test_grid_finds_room_again_through_other_instances(gpu):
    """A voxel put into another instance's cell takes the grid away; the other
    instance's voxel leaving brings it back, right, with the first untouched."""
    sc, acc = _load(20, 10, 0.4)
    insts, box = acc.read_instances(), acc.read_world()["aabbs"]
    assert len(insts) >= 3
    a, b = insts[0].first_primitive_index, insts[1].first_primitive_index
    old_a, old_b = box[a].copy(), box[b].copy()
    acc.update_blas(0, edits=[(0, old_b)])
    acc.update_scene()
    _same(acc, sc, 1, n=30000)
    acc.update_blas(2, edits=[(0, box[insts[2].first_primitive_index] + np.float32(1 / 32))])
    acc.update_scene()
    _same(acc, sc, 2, n=30000)
    acc.delete_primitive(1, 0)
    acc.update_scene()
    _same(acc, sc, 3, n=30000)
    acc.undo()
    acc.update_scene()
    _same(acc, sc, 4, n=30000)
    acc.update_blas(1, edits=[(0, old_a)])
    acc.update_scene()
    _same(acc, sc, 5, n=30000)
    acc.delete_blas(1)
    acc.update_scene()
    _same(acc, sc, 6, n=30000)


def test_grid_is_rebuilt_when_its_ids_run_out(gpu):
    """Instances that leave and come back take new ranges of ids each time,
    more in all than an update's reserve holds."""
    sc, acc = _load(40, 20, 0.5)
    assert len(acc.read_instances()) == 8
    for k in range(14):
        inst = k % 8
        r = acc.read_instances()[inst]
        W = acc.read_world()
        f, n = r.first_primitive_index, r.primitive_count
        boxes, prims = W["aabbs"][f:f + n].copy(), W["prims"][f:f + n].copy()
        acc.delete_blas(inst)
        acc.update_scene()
        _add_instance(acc, boxes, prims)
        acc.update_scene()
        print("in and out", k, flush=True)
        _same(acc, sc, 200 + k, n=12000)


def test_update_with_more_instances_than_the_grid_was_built_for(gpu):
    """One instance of 7000 slots gives way to 100 small ones in one update,
    in the same slots: nothing else of the scene is new."""
    d = ctamd.SceneDesc()
    d.grid[:] = [24, 24, 48]
    d.chunk[:] = [24] * 3
    d.occupied_count = 14000
    d.le_min = d.le_max = 1.0
    d.albedo_min, d.albedo_max = 0.2, 0.8
    d.seed = 9
    d.voxel_extent = ctamd.CT_VOXEL_EXTENT
    sc = ctamd.Scene(d)
    acc = ctamd.Accel(max_instances=200, max_primitives=sc.info.primitive_count + 20000, max_cube_lights=8)
    adj._load_geometry(sc, acc)
    _same(acc, sc, 1, n=20000)
    r = acc.read_instances()[0]
    W = acc.read_world()
    f = r.first_primitive_index
    assert r.primitive_count > 32 * 100
    boxes, prims = W["aabbs"][f:f + 3200].copy(), W["prims"][f:f + 3200].copy()
    acc.delete_blas(0)
    st = acc.staging()
    C.memmove(st.aabbs, boxes.ctypes.data, boxes.nbytes)
    C.memmove(st.primitives, prims.ctypes.data, prims.nbytes)
    t = ctamd.Task()
    t.type = ctamd.CT_TASK_BUILD_BLAS_FROM_CPU
    t.u.blas_build_from_cpu.instance_count = 100
    t.u.blas_build_from_cpu.primitive_count = 3200
    for k in range(16):
        t.u.blas_build_from_cpu.transform[k] = 1.0 if k % 5 == 0 else 0.0
    for k in range(100):
        st.instances[k].first_primitive_index = 32 * k
        st.instances[k].primitive_count = 32
    acc.task_queue_add(t)
    acc.update_scene()
    assert sum(i.primitive_count > 0 for i in acc.read_instances()) == 101
    _same(acc, sc, 2, n=20000)
    acc.delete_primitive(50, 3)
    acc.update_scene()
    _same(acc, sc, 3, n=20000)


def test_path_tracing_from_far_away_matches_oracle(gpu):
    """A far view beside a near one: path tracing asks about every view."""
    w = ctamd.hd_di(width=16, height=16, grid=32, chunk=16)
    sc = ctamd.Scene(ctamd.scene_desc(w))
    acc = ctamd.Accel(max_instances=sc.info.instance_count + 8,
                      max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024,
                      max_cube_lights=sc.info.cube_light_count + 8)
    ctx = ctamd.Ctx(16, 16)
    ctamd.load_scene(sc, acc, ctx)
    back = np.array([0.48, 0.6, 0.64])
    right = np.cross([0.0, 1.0, 0.0], back)
    right /= np.linalg.norm(right)
    far = 2e4
    views = adj.orbit_views(2, 160, 120, (0, 0, 0), 1.6, 0.4, fov_radians=1.2 / far)
    near = adj.orbit_views(1, 160, 120, (0, 0, 0), 1.6, 0.4)[0]
    views[0] = near
    m = np.zeros((4, 4))
    m[:3, 0], m[:3, 1], m[:3, 2], m[:3, 3], m[3, 3] = right, np.cross(back, right), back, far * back, 1.0
    views[1].inv_view[:] = np.float32(m.T.reshape(16)).tolist()
    img = adj.path_trace(acc, views, list(sc.materials), spp=2, max_depth=2, seed=5).cpu().numpy()
    osc = O.OScene.from_scene(sc)
    ref = osc.path_trace(ctamd.AdjointDesc(2, 2, 2, 5), views, list(sc.materials))
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    assert (img[:19200] != 0).any() and (img[19200:] != 0).any()
