"""Where the camera rays of a tile begin (tile_entry): no ray's closest hit is
another than from the whole scene. CPU build of the device code."""
import ctypes as C

import numpy as np
import pytest

import hostpath
from glslpt import scenes
from glslpt.renderer import options_for
from glslpt.scene import sphere_light


def tile_hits(sc, rs, cam, window, spp, **opts):
    """(rays whose hit differs, rays that hit, tiles that leave something out)
    in the tiles [x0, x1) x [y0, y1)."""
    o = options_for(rs, **opts)
    v = sc.view()
    tx, ty = (rs.width + 7) // 8, (rs.height + 7) // 8
    x0, y0, x1, y1 = window
    out = [C.c_int(0) for _ in range(3)]
    rc = hostpath.lib().host_tile_hits(C.byref(v), C.byref(o), C.byref(cam), max(x0, 0), max(y0, 0), min(x1, tx),
                                       min(y1, ty), spp, *(C.byref(c) for c in out))
    assert rc == 0
    return tuple(c.value for c in out)


def lights_in_view(rng, num, width, height, fov, ratio):
    """Three small meshes and `num` sphere lights of radius ratio * distance at
    random pixels of a view of `fov` degrees, half of them near a tile's border;
    also each light's pixel."""
    sc, rs = scenes.instanced_spheres(num_instances=3, freq=2, width=width, height=height, spp=16, max_depth=1)
    eye = np.array([3.0, 41.0, 307.0])
    sc.AddCamera(tuple(eye), (1.0, 2.0, 3.0), fov)
    cam = sc.camera()
    right, up, fwd = (np.array(list(getattr(cam, k)), np.float64) for k in ("right", "up", "forward"))
    s = np.tan(cam.fov * 0.5)
    at = []
    for k in range(num):
        px, py = rng.uniform(0, width), rng.uniform(0, height)
        if k & 1:
            px, py = 8 * round(px / 8) + rng.normal() * 0.3, 8 * round(py / 8) + rng.normal() * 0.3
        d = (2 * px / width - 1) * s * right + (2 * py / height - 1) * s * height / width * up + fwd
        dist = 10.0 ** rng.uniform(1, 4)
        pos = eye + d / np.linalg.norm(d) * dist
        sc.AddLight(sphere_light(tuple(float(x) for x in pos), float(ratio * dist), (1, 1, 1)))
        at.append((px, py))
    sc.ProcessScene()
    return sc, rs, cam, at


@pytest.mark.parametrize("ratio", [1e-2, 1e-3, 3e-4, 1e-4, 3e-5, 1e-5])
@pytest.mark.parametrize("width,height,fov", [(1920, 1080, 40.0), (3840, 2160, 40.0), (3840, 2160, 100.0),
                                              (1280, 720, 1.0), (1280, 720, 0.09)])
def test_distant_sphere_lights(ratio, width, height, fov):
    """The sphere test's float rounding accepts rays far outside a small distant
    sphere: the tiles of those rays keep their lights."""
    rng = np.random.default_rng(7)
    sc, rs, cam, at = lights_in_view(rng, 12, width, height, fov, ratio)
    differ = hits = 0
    for px, py in at:
        # half a window: the sphere, or what rounding adds to it, and two tiles more
        reach = int(max(ratio, 5e-4) * width / (2 * np.tan(cam.fov * 0.5)) / 8) + 2
        reach = min(reach, 24)
        tx, ty = int(px // 8), int(py // 8)
        d, h, _ = tile_hits(sc, rs, cam, (tx - reach, ty - reach, tx + reach + 1, ty + reach + 1), 16)
        differ += d
        hits += h
    print(f"{differ} of {hits} hits differ")
    assert hits > 0 and differ == 0


def test_lights_are_still_left_out():
    """A light of ordinary size is left out by most tiles."""
    sc, rs, cam, at = lights_in_view(np.random.default_rng(8), 1, 640, 360, 40.0, 0.02)
    differ, _, culled = tile_hits(sc, rs, cam, (0, 0, 80, 45), 1)
    assert differ == 0 and culled > 80 * 45 * 0.9


@pytest.mark.parametrize("width4", [2, 4])
@pytest.mark.parametrize("far", [0.0, 1e3, 1e5])
@pytest.mark.parametrize("freq", [0, 2])
def test_instance_boxes_are_tested(freq, far, width4):
    """Instances far from the origin, where the rounding of boxes and rays is
    seen at silhouettes: a tile that sees one instance alone tests its box all
    the same. freq 0: single quads, whose BLAS has no box of its own."""
    rng = np.random.default_rng(11)
    sc = scenes.Scene()
    if freq:
        mesh = sc.AddMesh(*scenes.displaced_icosphere(freq, 0.1, 3), name="sphere")
    else:
        mesh = sc.AddMesh(*scenes._uv_quad((-0.5, -0.5, 0), (1, 0, 0), (0, 1, 0)), name="quad")
    mat = sc.AddMaterial(baseColor=(0.7, 0.7, 0.7))
    for k in range(40):
        t = rng.uniform(-12, 12, 3) + np.array([far, -far, far])
        rot = scenes.random_rotation(rng) if k % 4 else np.eye(4)
        sc.AddMeshInstance(mesh, scenes.mat4(translate=t, scale=(rng.uniform(0.5, 3),) * 3, rot=rot), mat)
    sc.AddCamera((far, -far, far + 36), (far, -far, far), 45.0)
    sc.ProcessScene()
    rs = scenes.RenderSettings(400, 300, 16, 1)
    differ, hits, culled = tile_hits(sc, rs, sc.camera(), (0, 0, 50, 38), 16, bvh_width=width4)
    print(f"{differ} of {hits} hits differ, {culled} tiles culled")
    assert differ == 0 and hits > 1000 and culled > 100


@pytest.mark.parametrize("width4", [2, 4])
def test_boxes_with_swapped_planes(width4):
    """A TLAS whose boxes have their planes swapped on some axes, which the slab
    test takes as they are meant: the tiles do too."""
    rng = np.random.default_rng(12)
    sc, rs = scenes.instanced_spheres(num_instances=24, freq=3, width=160, height=96, spp=16, max_depth=1, extent=12.0)
    v, cam = sc.view(), sc.camera()
    nodes = np.ctypeslib.as_array(C.cast(v.nodes, C.POINTER(C.c_float)), (v.num_nodes, 9)).copy()
    swap = rng.random((v.num_nodes, 3)) < 0.5
    swap[:v.top_level_index] = False
    lo, hi = nodes[:, :3].copy(), nodes[:, 3:6].copy()
    nodes[:, :3], nodes[:, 3:6] = np.where(swap, hi, lo), np.where(swap, lo, hi)
    v.nodes = C.cast(nodes.ctypes.data, type(v.nodes))
    o = options_for(rs, bvh_width=width4)
    out = [C.c_int(0) for _ in range(3)]
    assert hostpath.lib().host_tile_hits(C.byref(v), C.byref(o), C.byref(cam), 0, 0, 20, 12, 16,
                                         *(C.byref(c) for c in out)) == 0
    differ, hits, culled = (c.value for c in out)
    print(f"{differ} of {hits} hits differ")
    assert differ == 0 and hits > 1000 and culled > 20
