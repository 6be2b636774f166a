"""Scenes that keep the BVH (two transforms, so no cell grid): path tracing."""
import numpy as np
import pytest

import ctamd
import oracle as O
from ctamd import adjoint as AD
from helpers import bits, oracle_scene_from_accel

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
