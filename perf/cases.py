"""The work that a user of this framework has it do, as measurable cases.

Each case goes through the public entry points of ``ctamd``: rendered ReSTIR
frames (single views and batches), plain path tracing, the differentiable
renderer, ray queries, interactive edits and acceleration-structure builds.
``listed()`` names the cases, ``draw()`` gives more of the same ranges.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube-tracing_amd"))

import ctamd  # noqa: E402
from ctamd import adjoint as adj  # noqa: E402
from ctamd.voxfile import monument  # noqa: E402

ORBIT = 360  # a closed camera orbit of 1 degree a frame


def listed():
    return [
        # A preview window on a small scene: a few short launches a frame, so
        # launch and host latency count.
        {"name": "frames_small", "kind": "frames", "scene": "noise", "grid": 64, "width": 256, "height": 256,
         "frames": 4, "depth": 1, "hybrid": False, "taa": True},
        # The benchmark's frame: 1080p, 4.2 M voxels, DI and 3-bounce ReSTIR PT,
        # a turntable of which the last frame is taken.
        {"name": "frames_hd", "kind": "frames", "scene": "noise", "grid": 256, "width": 1920, "height": 1080,
         "frames": 8, "depth": 3, "hybrid": False, "taa": True},
        # A large palette world with the hybrid shift and 4 bounces.
        {"name": "frames_palette", "kind": "frames", "scene": "palette", "grid": 384, "width": 1920, "height": 1080,
         "frames": 4, "depth": 4, "hybrid": True, "taa": True},
        # A MagicaVoxel model in an oddly sized window, direct light only.
        {"name": "frames_vox", "kind": "frames", "scene": "vox", "grid": 64, "width": 1277, "height": 717,
         "frames": 8, "depth": 0, "hybrid": False, "taa": True},
        # A server that renders many views of several scenes at once.
        {"name": "batch_16", "kind": "batch", "views": 16, "grid": 128, "min_side": 128, "max_width": 1024,
         "max_height": 768, "frames": 2, "depth": 2},
        # Unbiased reference images with metal, glass and media.
        {"name": "path_trace_hd", "kind": "path_trace", "grid": 256, "width": 1920, "height": 1080, "spp": 1,
         "depth": 3},
        # One step of inverse rendering: a small problem, then the full one
        # (8 views of 512^2 at 16 samples over 128^3).
        {"name": "fit_small", "kind": "fit", "grid": 48, "views": 2, "width": 96, "height": 80, "spp": 2, "depth": 2},
        {"name": "fit_large", "kind": "fit", "grid": 128, "views": 8, "width": 512, "height": 512, "spp": 16,
         "depth": 3},
        # Gradients of a rendered ReSTIR frame with respect to its materials.
        {"name": "frame_gradient", "kind": "frame_gradient", "grid": 160, "width": 1280, "height": 720, "depth": 2},
        # Ray queries from host arrays (picking, visibility, collision).
        {"name": "rays", "kind": "rays", "grid": 96, "rays": 100003},
        # An editing session: remove a voxel, look, take it back, look again.
        {"name": "edit", "kind": "edit", "grid": 128, "width": 960, "height": 540, "depth": 1, "edits": 2, "op": "delete"},
        # Loading a world: staging, BLAS and TLAS build, upload.
        {"name": "build", "kind": "build", "grid": 160, "chunk": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frames", "frames", "frames", "batch", "path_trace", "fit", "fit", "frame_gradient", "rays",
                       "edit", "build"])
    if kind == "frames":
        scene = rng.choice(["noise", "noise", "palette", "vox"])
        grid = {"noise": (24, 256), "palette": (64, 320), "vox": (24, 64)}[scene]
        return {"kind": kind, "scene": scene, "grid": _log(rng, *grid), "width": _log(rng, 97, 1920),
                "height": _log(rng, 64, 1080), "frames": rng.randint(2, 8),
                "depth": rng.randint(2, 4) if scene == "palette" else rng.randint(0, 3), "hybrid": scene == "palette",
                "taa": rng.random() < 0.8}
    if kind == "batch":
        return {"kind": kind, "views": rng.randint(2, 16), "grid": _log(rng, 32, 128), "min_side": 64,
                "max_width": _log(rng, 160, 1024), "max_height": _log(rng, 120, 768), "frames": rng.randint(1, 3),
                "depth": rng.randint(0, 3)}
    if kind == "path_trace":
        return {"kind": kind, "grid": _log(rng, 24, 256), "width": _log(rng, 65, 1920), "height": _log(rng, 65, 1080),
                "spp": rng.randint(1, 4), "depth": rng.randint(1, 6)}
    if kind == "fit":
        return {"kind": kind, "grid": _log(rng, 24, 128), "views": rng.randint(1, 8), "width": _log(rng, 33, 512),
                "height": _log(rng, 33, 512), "spp": _log(rng, 1, 16), "depth": rng.randint(1, 4)}
    if kind == "frame_gradient":
        return {"kind": kind, "grid": _log(rng, 32, 192), "width": _log(rng, 97, 1920), "height": _log(rng, 64, 1080),
                "depth": rng.randint(0, 3)}
    if kind == "rays":
        return {"kind": kind, "grid": _log(rng, 16, 192), "rays": _log(rng, 17, 400000)}
    if kind == "edit":
        return {"kind": kind, "grid": _log(rng, 32, 160), "width": _log(rng, 97, 1280), "height": _log(rng, 64, 720),
                "depth": rng.randint(0, 2), "edits": rng.randint(1, 3), "op": rng.choice(["delete", "move"])}
    return {"kind": kind, "grid": _log(rng, 32, 192), "chunk": rng.choice([32, 64])}


# --------------------------------------------------------------- preparation
def _noise_scene(grid, seed, fill=0.25, chunk=64, palette=(0, 0)):
    d = ctamd.SceneDesc()
    d.grid[:] = [grid] * 3
    d.chunk[:] = [min(chunk, grid)] * 3
    d.occupied_count = round(fill * grid ** 3)
    d.emissive_count = 0 if palette[0] else round(0.02 * d.occupied_count)
    d.le_min, d.le_max = 1.0, 20.0
    d.albedo_min, d.albedo_max = 0.2, 0.8
    d.seed = seed & 0xFFFFFFFF
    d.palette_size, d.palette_emissive = palette
    d.voxel_extent = ctamd.CT_VOXEL_EXTENT
    return ctamd.Scene(d)


def _scene(kind, grid, seed):
    if kind == "palette":
        return _noise_scene(grid, seed, fill=0.12, palette=(256, 3))
    if kind == "vox":
        return ctamd.Scene.from_vox(monument(n=grid, seed=seed % (1 << 31)), chunk=(64, 64, 64))
    return _noise_scene(grid, seed)


def _accel(sc):
    return ctamd.Accel(max_instances=sc.info.instance_count + 8,
                       max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024,
                       max_cube_lights=max(sc.info.cube_light_count, 1) + 8)


def _workload(sc, width, height, depth, hybrid=False, taa=True, start_deg=0.0):
    w = ctamd.vox_view(sc, width=width, height=height, indirect=depth > 0, max_depth=max(depth, 1), name="case")
    ext = float((sc.grid_max - sc.grid_min).max())
    mid = (sc.grid_min + sc.grid_max) / 2

    def camera(f):
        a = math.radians(start_deg + f)
        rel = np.array([1.5 * ext * math.sin(a), 0.375 * ext, 1.5 * ext * math.cos(a)])
        fwd = -rel / np.linalg.norm(rel)
        return tuple((mid + rel).tolist()), tuple(fwd.tolist()), (0.0, 1.0, 0.0)

    w.camera, w.taa = camera, taa
    if hybrid:
        w.restir.pt_shift_mapping = ctamd.CT_SHIFT_HYBRID
    return w


def _orbit(sc, case, seed):
    """The frame records of a closed orbit whose start the seed gives."""
    w = _workload(sc, case["width"], case["height"], case["depth"], case.get("hybrid", False), case.get("taa", True),
                  start_deg=float(seed % 360))
    return [ctamd.frame_params(w, f) for f in range(ORBIT + 1)]


def _views(sc, n, width, height, seed):
    ext = float((sc.grid_max - sc.grid_min).max())
    return adj.orbit_views(n, width, height, tuple(((sc.grid_min + sc.grid_max) / 2).tolist()), 1.6 * ext, 0.4 * ext,
                           start_deg=float(seed % 360))


def prepare(case, seed):
    return {"frames": _prepare_frames, "batch": _prepare_batch, "path_trace": _prepare_path_trace, "fit": _prepare_fit,
            "frame_gradient": _prepare_frame_gradient, "rays": _prepare_rays, "edit": _prepare_edit,
            "build": _prepare_build}[case["kind"]](case, seed)


def _prepare_frames(case, seed):
    sc = _scene(case["scene"], case["grid"], 0xC1 + seed)
    acc, ctx = _accel(sc), ctamd.Ctx(case["width"], case["height"])
    ctamd.load_scene(sc, acc, ctx)
    orbit = _orbit(sc, case, seed)
    ctx.render(acc, orbit[0])  # the program has been running: a previous frame exists
    return {"case": case, "scene": sc, "accel": acc, "ctx": ctx, "orbit": orbit, "at": 1}


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    scenes = []
    for k in range(4):
        sc = _noise_scene(max(16, case["grid"] >> (k % 2)), 0xC3 + 4 * seed + k, fill=float(rng.uniform(0.1, 0.3)))
        scenes.append([sc, _accel(sc), False])
    ctxs, accs, orbits = [], [], []
    # the sizes belong to the case: the seed moves the cameras and the scenes
    sizes = np.random.default_rng(case["views"])
    for v in range(case["views"]):
        sc, acc, loaded = scenes[v % 4]
        w = int(sizes.integers(case["min_side"], case["max_width"] + 1))
        h = int(sizes.integers(case["min_side"], case["max_height"] + 1))
        ctx = ctamd.Ctx(w, h)
        if loaded:
            ctamd.bind_scene(sc, ctx)
        else:
            ctamd.load_scene(sc, acc, ctx)
            scenes[v % 4][2] = True
        wl = _workload(sc, w, h, case["depth"], start_deg=float(rng.uniform(0, 360)))
        ctxs.append(ctx)
        accs.append(acc)
        orbits.append([ctamd.frame_params(wl, f) for f in range(41)])
    batch = ctamd.Batch(ctxs, accs)
    batch.render([o[0] for o in orbits])
    return {"case": case, "scenes": scenes, "ctxs": ctxs, "batch": batch, "orbits": orbits, "at": 1}


def _prepare_path_trace(case, seed):
    sc = _noise_scene(case["grid"], 0xC1 + seed)
    acc = _accel(sc)
    adj._load_geometry(sc, acc)
    mats = (ctamd.Material * sc.info.material_count).from_buffer_copy(sc.materials)
    a = np.frombuffer(mats, np.uint32).reshape(-1, 21)  # 84-byte MATERIAL records
    f = a.view(np.float32)
    f[:, 7:10] = f[:, 4:7]  # specular = diffuse
    for k, (kind, rough, ior) in enumerate([(ctamd.CT_MATERIAL_METAL, 0.3, 1.0), (ctamd.CT_MATERIAL_DIELECTRIC, 0.0, 1.5),
                                            (ctamd.CT_MATERIAL_CONSTANT_MEDIUM, 1.0, 1.0)]):
        a[4 * k + 3::12, 0] = kind
        f[4 * k + 3::12, 17] = rough
        f[4 * k + 3::12, 18] = ior
    views = _views(sc, 1, case["width"], case["height"], seed)
    one = _views(sc, 1, 8, 8, seed)
    adj.path_trace(acc, one, mats, 1, 1)  # uploads the materials, which stay in the accel
    return {"case": case, "accel": acc, "views": views, "seed": seed & 0xFFFF}


def _prepare_fit(case, seed):
    sc = _noise_scene(case["grid"], 0xC4 + seed, fill=0.24)
    acc = _accel(sc)
    adj._load_geometry(sc, acc)
    slots = adj.VoxelSlots(sc, acc)
    rng = np.random.default_rng(seed)
    n = sc.info.primitive_count
    lit = np.flatnonzero(rng.random(n) < 0.02)
    emission = np.zeros(n, np.float32)
    emission[lit] = rng.uniform(1.0, 20.0, lit.size)
    dev = torch.device("cuda")
    renderer = adj.DiffRenderer(acc, _views(sc, case["views"], case["width"], case["height"], seed), case["spp"],
                                case["depth"], 0xC4 + seed & 0xFFFF)

    room = n + 32 * (-(-case["grid"] // 64)) ** 3  # slots of any seed: ranges are aligned to 32

    def up(v):
        a = torch.zeros((room,) + v.shape[1:], dtype=torch.float32)
        a[:slots.capacity] = torch.from_numpy(slots.scatter(v))
        return a.to(dev)

    target = renderer.forward(up(rng.uniform(0.2, 0.8, (n, 3))), up(emission))
    return {"case": case, "accel": acc, "renderer": renderer, "target": target,
            "albedo": up(rng.uniform(0.2, 0.8, (n, 3))).requires_grad_(True),
            "emission": up(emission * rng.uniform(0.5, 1.5, n)).requires_grad_(True)}


def _prepare_frame_gradient(case, seed):
    s = _prepare_frames(dict(case, scene="noise"), seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    s["grad"] = torch.randn((case["width"] * case["height"], 4), generator=g, device="cuda", dtype=torch.float32)
    return s


def _rays_of(sc, n, seed):
    """Rays into the scene from around and from within it, host arrays."""
    rng = np.random.default_rng(seed)
    lo, hi = sc.grid_min.astype(np.float64), sc.grid_max.astype(np.float64)
    ext = (hi - lo).max()
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    inside = rng.random(n) < 0.5
    to = rng.uniform(lo, hi, (n, 3))
    o = np.where(inside[:, None], to, to - d * (1.5 * ext))
    dist = np.where(inside, rng.uniform(0.05, 0.5, n), 1.5) * ext
    return (np.ascontiguousarray(o, np.float32), np.ascontiguousarray(d, np.float32),
            np.ascontiguousarray(dist, np.float32))


def _prepare_rays(case, seed):
    sc = _noise_scene(case["grid"], 0xA1 + seed, fill=0.15)
    acc = _accel(sc)
    adj._load_geometry(sc, acc)
    o, d, dist = _rays_of(sc, case["rays"], seed)
    return {"case": case, "accel": acc, "o": o, "d": d, "dist": dist}


def _prepare_edit(case, seed):
    s = _prepare_frames(dict(case, scene="noise"), seed)
    rng = np.random.default_rng(seed)
    sc, acc = s["scene"], s["accel"]
    s["edit"] = []
    for _ in range(case["edits"]):
        inst = int(rng.integers(0, sc.info.instance_count))
        s["edit"].append((inst, int(rng.integers(0, sc.instances[inst].primitive_count))))
    s["accel"].update_scene()  # the load has settled
    return s


def _prepare_build(case, seed):
    sc = _noise_scene(case["grid"], 0xB1 + seed, chunk=case["chunk"])
    o, d, _ = _rays_of(sc, 20000, seed)
    return {"case": case, "scene": sc, "o": o, "d": d}


# --------------------------------------------------------------------- run
def run(state):
    return {"frames": _run_frames, "batch": _run_batch, "path_trace": _run_path_trace, "fit": _run_fit,
            "frame_gradient": _run_frame_gradient, "rays": _run_rays, "edit": _run_edit,
            "build": _run_build}[state["case"]["kind"]](state)


def _next(s, n):
    """The next frame record of the orbit (frame 0 only starts it)."""
    f = s["at"]
    s["at"] = f + 1 if f < n else 1
    return f


def _run_frames(s):
    c, ctx, acc, orbit = s["case"], s["ctx"], s["accel"], s["orbit"]
    for _ in range(c["frames"]):
        ctx.render(acc, orbit[_next(s, ORBIT)])
    return ctx.read(ctamd.CT_BUF_IMAGE, c["width"], c["height"])


def _run_batch(s):
    for _ in range(s["case"]["frames"]):
        f = _next(s, 40)
        s["batch"].render([o[f] for o in s["orbits"]])
    return [ctx.read(ctamd.CT_BUF_IMAGE, o[0].width, o[0].height) for ctx, o in zip(s["ctxs"], s["orbits"])]


def _run_path_trace(s):
    c = s["case"]
    return adj.path_trace(s["accel"], s["views"], None, c["spp"], c["depth"], s["seed"])


def _run_fit(s):
    image = adj.render(s["renderer"], s["albedo"], s["emission"])
    loss = ((image - s["target"]) ** 2).mean()
    ga, ge = torch.autograd.grad(loss, [s["albedo"], s["emission"]])
    return {"image": image, "albedo": ga, "emission": ge}


def _run_frame_gradient(s):
    ctx, acc = s["ctx"], s["accel"]
    p = s["orbit"][_next(s, ORBIT)]
    ctx.render(acc, p)
    gd, ge = adj.frame_adjoint(ctx, acc, p, s["grad"], s["scene"].info.material_count)
    return {"diffuse": gd, "emission": ge}


def _run_rays(s):
    acc, o, d = s["accel"], s["o"], s["d"]
    t, ids = acc.trace_closest(o, d)
    b = acc.trace_bounce(o, d)
    return {"t": t, "ids": ids, "occluded": acc.trace_any(o, d, s["dist"]), "bounce_ids": b["ids"], "pos": b["pos"],
            "nrm": b["nrm"], "dist": b["dist"]}


def _run_edit(s):
    c, ctx, acc = s["case"], s["ctx"], s["accel"]

    def look():
        p = ctamd.FrameParams.from_buffer_copy(s["orbit"][_next(s, ORBIT)])
        if acc.remapping_active():
            p.is_active |= ctamd.CT_REMAP_BIT
        ctx.render(acc, p)
        # shown before the next edit, which may not touch a scene in use
        return ctx.read(ctamd.CT_BUF_IMAGE, c["width"], c["height"])

    images = []
    for k, (inst, prim) in enumerate(s["edit"]):
        if c["op"] == "delete":
            acc.delete_primitive(inst, prim)
        else:
            acc.update_blas(inst, transform=_shift(0.125 * (k + 1)))
        acc.update_scene()
        images.append(look())
        if c["op"] == "delete":
            acc.undo()
        else:
            acc.update_blas(inst, transform=_shift(-0.125 * (k + 1)))
        acc.update_scene()
        images.append(look())
    return images


def _shift(dx):
    m = np.eye(4, dtype=np.float32)
    m[3, 0] = dx  # column-major: column 3 is the translation
    return m.reshape(16)


def _run_build(s):
    sc = s["scene"]
    acc, ctx = _accel(sc), ctamd.Ctx(16, 16)
    ctamd.load_scene(sc, acc, ctx)
    t, ids = acc.trace_closest(s["o"], s["d"])  # the first queries of the loaded world
    acc.close()
    ctx.close()
    return {"t": t, "ids": ids}


# ----------------------------------------------------------- work and error
def work(case):
    """Bytes: a frame reads the previous state of each pixel (64 of DI, 36 of
    reservoir, 96 of path reservoir, 16 of image) and writes the next; the
    image then goes to the host.  Operations: about 60 for each light
    candidate or box test that each sample cannot do without."""
    k = case["kind"]
    if k in ("frames", "batch", "edit", "frame_gradient"):
        if k == "batch":
            sizes = np.random.default_rng(case["views"])
            px = sum(int(sizes.integers(case["min_side"], case["max_width"] + 1)) *
                     int(sizes.integers(case["min_side"], case["max_height"] + 1)) for _ in range(case["views"]))
        else:
            px = case["width"] * case["height"]
        frames = {"frames": case.get("frames"), "batch": case.get("frames"), "edit": 2 * case.get("edits", 0),
                  "frame_gradient": 1}[k]
        state = 2 * (64 + 36 + 16 + (96 if case["depth"] else 0))
        out = 16 * px
        if k == "frame_gradient":
            out += 24 * round(0.25 * case["grid"] ** 3)
        return {"bytes": frames * px * state + out, "flops": frames * px * 60.0 * (32 + 4 + case["depth"])}
    if k == "path_trace":
        px = case["width"] * case["height"]
        return {"bytes": 12.0 * px, "flops": 60.0 * px * case["spp"] * (1 + case["depth"])}
    if k == "fit":
        px = case["views"] * case["width"] * case["height"]
        return {"bytes": 5 * 12.0 * px + 32.0 * round(0.24 * case["grid"] ** 3),
                "flops": 2 * 60.0 * px * case["spp"] * (1 + case["depth"])}
    if k == "rays":
        return {"bytes": case["rays"] * (24.0 + 12 + 24 + 48 + 28 + 1), "flops": 3 * 60.0 * case["rays"]}
    n = round(0.25 * case["grid"] ** 3)
    return {"bytes": n * (24.0 + 8 + 84 + 16 + 64), "flops": 60.0 * n}


def tolerance(case):
    """Every traversal, shading and sampling result is defined to the bit
    (single IEEE operations in a fixed order); only sums over paths and
    pixels that share a voxel are added in any order (two runs differ by
    1e-7 of the norm and 3e-6 of a value)."""
    if case["kind"] == "fit":
        return {"rel": 1e-6, "max": 2e-5}
    if case["kind"] == "frame_gradient":
        return {"rel": 5e-7, "max": 2e-5}
    return "exact"


def exact(case, seed):
    """Ray queries (and the first ones of a loaded world): the closest hit
    distance by brute force over every voxel in 64 bits.  The other kinds
    sample random paths and reservoirs whose branches a wider type takes
    differently, so they have no such value."""
    if case["kind"] == "build":
        sc = _noise_scene(case["grid"], 0xB1 + seed, chunk=case["chunk"])
        o, d, _ = _rays_of(sc, 20000, seed)
    elif case["kind"] == "rays":
        sc = _noise_scene(case["grid"], 0xA1 + seed, fill=0.15)
        o, d, _ = _rays_of(sc, case["rays"], seed)
    else:
        return None
    box = torch.from_numpy(sc.aabbs).to("cuda", torch.float64)
    if box.shape[0] * o.shape[0] > 1.5e10:
        return None
    o, d = (torch.from_numpy(v).to("cuda", torch.float64) for v in (o, d))
    best = torch.full((o.shape[0],), float("inf"), dtype=torch.float64, device="cuda")
    step = max(1, int(3e7 // box.shape[0]))
    for a in range(0, o.shape[0], step):
        oo, dd = o[a:a + step, None, :], d[a:a + step, None, :]
        near = far = None
        for k in range(3):
            t0, t1 = (box[None, :, k] - oo[..., k]) / dd[..., k], (box[None, :, 3 + k] - oo[..., k]) / dd[..., k]
            lo, hi = torch.minimum(t0, t1), torch.maximum(t0, t1)
            near = lo if near is None else torch.maximum(near, lo)
            far = hi if far is None else torch.minimum(far, hi)
        t = torch.where(near > 0, near, far)  # from within a voxel: where the ray leaves it
        t = torch.where((near <= far) & (far > 0), t, torch.inf)
        best[a:a + step] = t.min(dim=1).values
    t = torch.where(torch.isinf(best), -1.0, best)
    if case["kind"] == "build":
        return {"t": t, "ids": None}
    return {"t": t, "ids": None, "occluded": None, "bounce_ids": None, "pos": None, "nrm": None, "dist": None}
