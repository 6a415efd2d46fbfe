"""k_finish, the launch that runs the rest of a pass's paths to their end: a
pass run whole, a pass taken over after some staged bounces and a pass staged
to the end (compact_every 2) give the plain form's image bit for bit."""
import numpy as np
import pytest

from glslpt import scenes
from glslpt._capi import PT_MODE_PLAIN, PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


def image(r, sc, rs, mode, spp, **kw):
    r.set_options(options_for(rs, mode=mode, **kw))
    r.set_camera(sc.camera())
    r.clear()
    r.render(1, spp)
    r.synchronize()
    return r.read_accum()


@pytest.mark.parametrize("kind", ["envmap", "textures", "media", "volmis", "alpha_mask", "alpha_blend"])
def test_staged_then_finished(renderer, kind):
    """9.6M paths per pass: above the size that k_finish runs whole, so bounces
    are staged until few paths are left; compact_every 2 stages every bounce."""
    sc, rs = scenes.feature_scene(kind, width=1021, height=1033, spp=9, max_depth=6)
    renderer.upload_scene(sc)
    want = image(renderer, sc, rs, PT_MODE_PLAIN, 9)
    renderer.reset_stats()
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 9, wave_spp=9, bvh_width=4, extend_cap=16)
    ms = renderer.stats()["ms_stage"]
    assert ms["extend"] > 0 and ms["plain"] > 0
    assert np.isfinite(want).all()
    if kind != "alpha_blend":  # four-wide nodes can decide exact ties differently; blending walks BVH2 either way
        want4 = image(renderer, sc, rs, PT_MODE_PLAIN, 9, bvh_width=4)
        assert np.array_equal(got, want4)
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 9, wave_spp=9)
    assert np.array_equal(got, want)
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 9, wave_spp=9, compact_every=2)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("size", [(1, 1), (9, 1), (8, 8), (63, 65), (200, 117), (1030, 515)])
@pytest.mark.parametrize("depth", [0, 1, 7])
def test_whole_pass(renderer, size, depth):
    """Passes run whole, from one 8x8 tile (one path per wave) to full waves."""
    sc, rs = scenes.feature_scene("media", width=size[0], height=size[1], spp=3, max_depth=depth)
    renderer.upload_scene(sc)
    want = image(renderer, sc, rs, PT_MODE_PLAIN, 3)
    renderer.reset_stats()
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 3, wave_spp=2)
    ms = renderer.stats()["ms_stage"]
    assert ms["extend"] == 0 and ms["plain"] > 0
    assert np.array_equal(got, want)
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 3, wave_spp=2, compact_every=3)
    assert np.array_equal(got, want)


def test_adjoint_of_a_pass_run_whole(renderer):
    """The primal pass records the visible NEE rays wherever it runs: the
    gradient of a pass run whole equals that of one staged to the end."""
    sc, rs = scenes.material_boxes(num_boxes=24, sphere_freq=6, num_spheres=2, num_materials=8, width=72, height=40,
                                   spp=4, max_depth=5)
    renderer.upload_scene(sc)
    dl = np.random.default_rng(5).normal(size=(40, 72, 3)).astype(np.float32) / (40 * 72)
    g = []
    for cadence in (1, 2):
        renderer.set_options(options_for(rs, wave_spp=4, compact_every=cadence))
        renderer.set_camera(sc.camera())
        g.append(renderer.adjoint(0, 4, dl).astype(np.float64))
    # the same terms in another order of the float sums
    assert np.abs(g[0]).max() > 0
    assert np.abs(g[0] - g[1]).max() <= 1e-5 * np.abs(g[1]).max()
