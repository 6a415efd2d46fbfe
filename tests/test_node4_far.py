"""Scenes with boxes whose planes lie so far out that an entry or exit distance
is infinite (an instance moved to the end of the float range, to hide it): the
four-wide form finds the hits that the binary one finds. CPU build of the device
code."""
import ctypes as C

import numpy as np
import pytest

import hostpath
from common import random_dirs
from glslpt import scenes
from glslpt.renderer import options_for


def closest(sc, rs, o, d, **opts):
    v, opt, cam = sc.view(), options_for(rs, **opts), sc.camera()
    n = o.shape[0]
    t, tri, inst = np.zeros(n, np.float32), np.zeros(n, np.int32), np.zeros(n, np.int32)
    f, i = C.POINTER(C.c_float), C.POINTER(C.c_int)
    rc = hostpath.lib().host_closest(C.byref(v), C.byref(opt), C.byref(cam), n, o.ctypes.data_as(f),
                                     d.ctypes.data_as(f), t.ctypes.data_as(f), tri.ctypes.data_as(i),
                                     inst.ctypes.data_as(i))
    assert rc == 0
    return t, tri, inst


def hidden_scene(far, num=24):
    """Spheres within 5 units of the origin, every sixth moved to +-far on all axes."""
    rng = np.random.default_rng(3)
    sc = scenes.Scene()
    mesh = sc.AddMesh(*scenes.displaced_icosphere(3, 0.1, 3), name="sphere")
    mat = sc.AddMaterial(baseColor=(0.7, 0.7, 0.7))
    for k in range(num):
        at = rng.uniform(-5, 5, 3)
        if k % 6 == 0:
            at = far * rng.choice([-1.0, 1.0], 3)
        sc.AddMeshInstance(mesh, scenes.mat4(translate=at), mat)
    sc.AddCamera((0, 0, 20), (0, 0, 0), 45.0)
    sc.ProcessScene()
    return sc, scenes.RenderSettings(64, 64, 1, 2)


@pytest.mark.parametrize("far", [20.0, 1e17, 1e19, 1e30, 3.4e38])
@pytest.mark.parametrize("scale", [1.0, 1e-5])
def test_far_instances(far, scale):
    sc, rs = hidden_scene(far)
    rng = np.random.default_rng(4)
    n = 50000
    o = rng.uniform(-8, 8, (n, 3)).astype(np.float32)
    d = (random_dirs(rng, n) * np.float32(scale)).astype(np.float32)
    two, four = (closest(sc, rs, o, d, bvh_width=w) for w in (2, 4))
    hits = int((two[1] >= 0).sum())
    print(f"{hits} hits, {int((two[1] != four[1]).sum())} differ")
    for a, b in zip(two, four):
        assert np.array_equal(a, b)
    if scale == 1.0:  # a distance of 1e6 directions is as far as closest hits go
        assert hits > n // 10
