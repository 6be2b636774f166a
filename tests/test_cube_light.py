"""The cube light's draw (csrc/cube_light.h), built for the host, against the
text that computes every draw's point: the same outcome, random state, point
and ray origin to the bit."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("clang++")) if c and os.path.exists(c)), None)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if CLANG is None:
        pytest.skip("no clang++ (the device header uses its vector types)")
    out = str(tmp_path_factory.mktemp("light") / "liblight.so")
    src = os.path.join(HERE, "host_walk")
    subprocess.run([CLANG, "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-I", src, "-o", out,
                    os.path.join(src, "cube_light_host.cpp")], check=True)
    return C.CDLL(out)


@pytest.mark.parametrize("place", ["far", "near", "level", "inside", "origin"])
@pytest.mark.parametrize("normal", ["axis", "any"])
def test_draw_equals_the_text(lib, place, normal):
    rng = np.random.default_rng(["far", "near", "level", "inside", "origin"].index(place) * 2 + (normal == "any"))
    n = 200000
    size = np.where(rng.random(n) < 0.7, 0.03125, rng.uniform(0.01, 2.0, n))
    c = np.round(rng.uniform(-8, 8, (n, 3)) * 32) / 32 + 1 / 64
    if place == "origin":  # cells at the coordinate planes, where the ray origin takes its other branch
        c = rng.choice([-1, 0, 1], (n, 3)) / 32 + rng.choice([0, 1 / 64], (n, 3))
    nor = rng.normal(size=(n, 3))
    nor /= np.linalg.norm(nor, axis=1, keepdims=True)
    if normal == "axis":
        nor = np.eye(3)[rng.integers(0, 3, n)] * rng.choice([-1.0, 1.0], (n, 1))
        nor = np.where((nor == 0) & (rng.random((n, 3)) < 0.2), -0.0, nor)
    off = rng.uniform(-8, 8, (n, 3))
    if place in ("near", "origin"):
        off = rng.uniform(-2, 2, (n, 3)) * size[:, None]
    elif place == "inside":
        off = rng.uniform(-0.5, 0.5, (n, 3)) * size[:, None]
    elif place == "level":  # the planes of the voxel's faces and of the margin, or just beside them
        a = rng.integers(0, 3, n)
        at = rng.choice([-0.5, 0.5], n) * size + rng.choice([0, 1e-4, -1e-4, 1e-7, 9.9e-5, 1.1e-4], n)
        off[np.arange(n), a] = at
    P = c + off
    f32 = [np.ascontiguousarray(v, np.float32) for v in (P, nor, c, size)]
    seed = rng.integers(0, 1 << 32, n, dtype=np.uint32)
    taken = np.zeros(3, np.uint32)
    p = [v.ctypes.data_as(C.c_void_p) for v in f32 + [seed, taken]]
    assert lib.draws_differ(n, *p) == 0
    if place != "inside":
        assert taken[0] > n // 20
