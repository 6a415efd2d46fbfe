"""Camera rays that begin at their tile's TLAS entry (calls of ten samples and
more) against rays that begin at the root (calls of one sample): the same image
bit for bit, in every form."""
import numpy as np
import pytest

from glslpt import scenes
from glslpt._capi import PT_MODE_PLAIN, PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for
from glslpt.scene import quad_light, sphere_light

pytestmark = pytest.mark.gpu
SPP = 10


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


def compare(r, sc, rs, cam, **kw):
    for mode in (PT_MODE_PLAIN, PT_MODE_WAVEFRONT):
        for width in (2, 4):
            for cadence in ((1,) if mode == PT_MODE_PLAIN else (1, 2)):
                r.set_options(options_for(rs, mode=mode, bvh_width=width, wave_spp=SPP, compact_every=cadence, **kw))
                r.set_camera(cam)
                r.clear()
                r.render(0, SPP)
                r.synchronize()
                got = r.read_accum()
                r.clear()
                for s in range(SPP):
                    r.render(s, 1)
                r.synchronize()
                want = r.read_accum()
                assert np.array_equal(got, want, equal_nan=True), (mode, width, cadence)
    return got


def spheres(seed=5, **kw):
    args = dict(num_instances=24, freq=6, seed=seed, width=141, height=77, spp=SPP, max_depth=3, extent=12.0)
    args.update(kw)
    return scenes.instanced_spheres(**args)


VIEWS = {
    "outside": ((0, 6, 36), (0, 0, 0), 45.0),
    "inside": ((0.3, 0.2, 0.1), (4, 1, -3), 75.0),
    "away": ((0, 6, 36), (0, 6, 80), 45.0),
    "grazing": ((0, 0.0, 200.0), (14.0, 3.0, 0), 10.0),
    "tiny fov": ((0, 40, 300), (1.0, 2.0, 3.0), 0.05),
    "wide": ((0, 3, 14), (0, 0, 0), 150.0),
    "along an axis": ((0, 0, 30), (0, 0, 0), 30.0),
}


@pytest.mark.parametrize("view", VIEWS)
def test_views(renderer, view):
    sc, rs = spheres()
    renderer.upload_scene(sc)
    eye, at, fov = VIEWS[view]
    sc.AddCamera(eye, at, fov)
    compare(renderer, sc, rs, sc.camera())


@pytest.mark.parametrize("size", [(1, 1), (8, 8), (9, 17), (640, 3), (3, 640)])
def test_sizes(renderer, size):
    sc, rs = spheres(width=size[0], height=size[1])
    renderer.upload_scene(sc)
    compare(renderer, sc, rs, sc.camera())


def test_lens_and_far_coordinates(renderer):
    """A lens of positive radius keeps the root; a scene 1e5 units from the
    origin still loses no hit to rounding."""
    sc, rs = spheres()
    renderer.upload_scene(sc)
    cam = sc.camera()
    cam.aperture = 0.3
    cam.focalDist = 30.0
    compare(renderer, sc, rs, cam)
    xf = sc.arrays()["transforms"].copy()
    xf[:, 12] += 1e5
    xf[:, 13] -= 1e5
    renderer.rebuild_instances(xf)
    sc.AddCamera((1e5, -1e5 + 6, 36), (1e5, -1e5, 0), 45.0)
    img = compare(renderer, sc, rs, sc.camera())
    assert len(np.unique(img[..., 0])) > 10  # geometry is seen


def test_lights_in_the_view(renderer):
    """Only lights in the upper half of the view: a sphere, a rectangle and a
    rectangle whose sides are not at right angles."""
    sc, rs = spheres(num_instances=3)
    sc.AddLight(sphere_light((-9, 9, 0), 1.5, (3, 2, 1)))
    sc.AddLight(quad_light((0, 8, 0), (2, 8, 0), (0, 10, 0), (1, 2, 3)))
    sc.AddLight(quad_light((5, 8, 0), (8, 8, 0), (7, 10, 0), (2, 2, 2)))
    sc.ProcessScene()
    renderer.upload_scene(sc)
    sc.AddCamera((0, 8, 30), (0, 8, 0), 50.0)
    for hide in (0, 1):
        compare(renderer, sc, rs, sc.camera(), hide_emitters=hide)


@pytest.mark.parametrize("kind", ["envmap", "media", "alpha_blend", "volmis"])
def test_features(renderer, kind):
    sc, rs = scenes.feature_scene(kind, width=120, height=90, spp=SPP)
    renderer.upload_scene(sc)
    sc.AddCamera((0.0, 6.0, 14.0), (3.0, 4.0, 0.0), 60.0)  # half of the view is empty
    compare(renderer, sc, rs, sc.camera())


@pytest.mark.parametrize("mode", [PT_MODE_PLAIN, PT_MODE_WAVEFRONT])
def test_batch(renderer, mode):
    """Jobs of a batch whose mean samples reach the bound, one with a lens."""
    sc, rs = spheres()
    renderer.upload_scene(sc)
    jobs = []
    for k, (eye, at, fov) in enumerate(VIEWS.values()):
        sc.AddCamera(eye, at, fov)
        cam = sc.camera()
        if k == 1:
            cam.aperture = 0.2
        jobs.append(dict(camera=cam, width=65 + 8 * k, height=40 + k, spp=SPP + k, max_depth=1 + k))
    renderer.set_options(options_for(rs, mode=mode, wave_spp=4, use_graph=1, bvh_width=4))
    out = renderer.batch_render(jobs)
    for job, got in zip(jobs, out):
        renderer.set_options(options_for(rs, mode=mode, bvh_width=4, width=job["width"], height=job["height"],
                                         max_depth=job["max_depth"]))
        renderer.set_camera(job["camera"])
        renderer.clear()
        for s in range(job["spp"]):
            renderer.render(s, 1)
        renderer.synchronize()
        assert np.array_equal(got, renderer.read_accum())
