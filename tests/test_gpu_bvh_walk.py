"""Scenes that keep the BVH (two transforms, so no cell grid): path tracing,
the adjoint, frames with the RIS BRDF strategy and the hybrid shift, and
batches that mix such a scene with one walked through its grid."""
import numpy as np
import pytest

import ctamd
import oracle as O
from ctamd import adjoint as AD
from helpers import all_buffers_equal, bits, oracle_scene_from_accel

pytestmark = pytest.mark.gpu


def _shift_one(acc, dx=0.01171875):
    """Moves the last instance by 3/8 of a voxel."""
    m = np.eye(4, dtype=np.float32)
    m[3, 0] = dx
    acc.update_blas(len(acc.read_instances()) - 1, transform=m.reshape(16))
    acc.update_scene()
    acc.update_scene()  # settled


def _accel(sc):
    return ctamd.Accel(max_instances=sc.info.instance_count + 8,
                       max_primitives=sc.info.primitive_count + 32 * sc.info.instance_count + 1024,
                       max_cube_lights=max(sc.info.cube_light_count, 1) + 8)


def _mixed_materials(sc, seed=5):
    rng = np.random.default_rng(seed)
    mats = []
    for k, m0 in enumerate(sc.materials):
        m = ctamd.Material.from_buffer_copy(bytes(m0))
        m.type = k % 4
        if m.type == ctamd.CT_MATERIAL_METAL:
            m.specular[:] = m.diffuse[:]
            m.roughness = float(rng.uniform(0.0, 1.0))
        elif m.type == ctamd.CT_MATERIAL_DIELECTRIC:
            m.ior = float(rng.uniform(1.1, 1.8))
        mats.append(m)
    return mats


@pytest.mark.parametrize("width,height,spp,depth", [(37, 21, 1, 1), (64, 40, 3, 5), (1, 1, 7, 7)])
def test_path_trace_matches_oracle(gpu, width, height, spp, depth):
    w = ctamd.hd_di(width=width, height=height, grid=48, chunk=16, max_depth=2)
    sc = ctamd.Scene(ctamd.scene_desc(w))
    acc, ctx = _accel(sc), ctamd.Ctx(8, 8)
    ctamd.load_scene(sc, acc, ctx)
    _shift_one(acc)
    mats = _mixed_materials(sc)
    extent = 48 * ctamd.CT_VOXEL_EXTENT
    views = AD.orbit_views(2, width, height, (0, 0, 0), 1.6 * extent, 0.4 * extent)
    print("bvh path trace", width, height, spp, depth, flush=True)
    img = AD.path_trace(acc, views, mats, spp=spp, max_depth=depth, seed=0x77).cpu().numpy()
    osc, _, _ = oracle_scene_from_accel(acc, list(sc.materials), ctx.light_config())
    ref = osc.path_trace(ctamd.AdjointDesc(len(views), spp, depth, 0x77), views, mats)
    assert np.array_equal(bits(img), bits(ref))
    assert np.isfinite(img).all() and (img.any() or width * height == 1)


@pytest.mark.parametrize("depth", [0, 3, 5, 6, 7])
def test_adjoint_matches_oracle(gpu, depth):
    """Depths on both sides of where the backward pass keeps a path's vertices
    elsewhere."""
    import torch
    w = AD.AdjointWorkload(grid=48, chunk=16, width=40, height=31, views=2, spp=3, max_depth=depth)
    sc, alb, emi = AD.build_scene(w)
    acc = _accel(sc)
    AD._load_geometry(sc, acc)
    slots = AD.VoxelSlots(sc, acc)
    _shift_one(acc)
    extent = w.grid * ctamd.CT_VOXEL_EXTENT
    views = AD.orbit_views(w.views, w.width, w.height, (0, 0, 0), 1.6 * extent, 0.4 * extent)
    r = AD.DiffRenderer(acc, views, w.spp, w.max_depth, w.target_seed)
    a, e = slots.scatter(alb), slots.scatter(emi)
    dev = torch.device("cuda")
    a_t, e_t = torch.from_numpy(a).to(dev), torch.from_numpy(e).to(dev)
    print("bvh adjoint", depth, flush=True)
    img = r.forward(a_t, e_t).cpu().numpy()
    osc, _, _ = oracle_scene_from_accel(acc, list(sc.materials), O.light_config_for(0, 0, 0))
    desc = ctamd.AdjointDesc(len(views), w.spp, w.max_depth, w.target_seed)
    n = len(acc.read_world()["aabbs"])  # the oracle's voxels are the accel's slots
    ref = osc.adjoint_render(desc, views, a[:n], e[:n])
    assert np.array_equal(bits(img), bits(ref))
    g = np.random.default_rng(3).normal(size=ref.shape).astype(np.float32)
    ga, ge = (v.cpu().numpy()[:n] for v in r.backward(a_t, e_t, torch.from_numpy(g).to(dev)))
    oga, oge = osc.adjoint_backward(desc, views, a[:n], e[:n], g)
    # sums of 32-bit terms in another order than the oracle's, in 64 bits
    assert np.allclose(ge, oge, rtol=1e-4, atol=1e-6 * np.abs(oge).max())
    assert np.allclose(ga, oga, rtol=1e-4, atol=1e-6 * max(np.abs(oga).max(), 1e-30))
    assert np.abs(oge).sum() > 0


def _loaded(w, shift):
    sc = ctamd.Scene(ctamd.scene_desc(w))
    acc, first = _accel(sc), ctamd.Ctx(8, 8)
    ctamd.load_scene(sc, acc, first)  # the accel holds the scene; contexts bind to it
    if shift:
        _shift_one(acc)
    return sc, acc


def _ctx(sc, w):
    ctx = ctamd.Ctx(w.width, w.height)
    ctamd.bind_scene(sc, ctx)
    return ctx


@pytest.mark.parametrize("kind", ["plain", "ris_brdf", "hybrid", "hybrid_ris_brdf"])
def test_frames_match_oracle(gpu, kind):
    w = ctamd.hd_di(width=57, height=35, grid=48, chunk=16, frames=3, max_depth=3)
    if "hybrid" in kind:
        w.restir.pt_shift_mapping = ctamd.CT_SHIFT_HYBRID
    if "brdf" in kind:
        w.features |= ctamd.CT_RIS_BRDF_BIT
        w.emissive *= 10
    sc, acc = _loaded(w, True)
    ctx = _ctx(sc, w)
    osc, _, _ = oracle_scene_from_accel(acc, list(sc.materials), ctx.light_config())
    ofr = O.OFrame(osc, w.width, w.height)
    for f in range(3):
        print("bvh frame", kind, f, flush=True)
        p = ctamd.frame_params(w, f)
        ctx.render(acc, p)
        ofr.render(p)
        hit = all_buffers_equal(ctx, ofr, w, f)
        assert hit.any() and not hit.all()


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_of_bvh_and_grid_scenes(gpu, use_graph):
    """Views of a scene with a cell grid beside views of one without, in one
    batch (which walks BVHs then), with the hybrid shift and the RIS BRDF
    strategy in some of them: each view's bits equal its own render."""
    scenes, views = ctamd.batched_views(n_views=6, seed=0xC3, grids=(48, 64), max_depth=2, size_scale=0.08)
    built = [_loaded(s, k == 0) for k, s in enumerate(scenes)]
    for n, (k, w) in enumerate(views):
        w.restir = ctamd.RestirParams.from_buffer_copy(bytes(w.restir))
        if n % 3 == 0:
            w.restir.pt_shift_mapping = ctamd.CT_SHIFT_HYBRID
        if n % 2 == 0:
            w.features |= ctamd.CT_RIS_BRDF_BIT
    assert {k for k, _ in views} >= {0, 1}
    plain = [_ctx(built[k][0], w) for k, w in views]
    batch_ctx = [_ctx(built[k][0], w) for k, w in views]
    b = ctamd.Batch(batch_ctx, [built[k][1] for k, _ in views])
    for f in range(3):
        print("mixed batch", use_graph, f, flush=True)
        ps = [ctamd.frame_params(w, f) for _, w in views]
        b.render(ps, use_graph=use_graph)
        for (k, w), ctx, p in zip(views, plain, ps):
            ctx.render(built[k][1], p)
        for n, ((k, w), pc, bc) in enumerate(zip(views, plain, batch_ctx)):
            for which in (ctamd.CT_BUF_IMAGE, ctamd.CT_BUF_DI, ctamd.CT_BUF_TEMPORAL_PATH_RESERVOIR):
                assert bytes(pc.read(which, w.width, w.height)) == bytes(bc.read(which, w.width, w.height)), (f, n, which)
