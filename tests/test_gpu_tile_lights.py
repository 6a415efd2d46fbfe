"""Small distant sphere lights, which the sphere test's rounding makes larger
than they are: a call of ten samples (camera rays begin at their tiles'
entries) gives the image of ten calls of one, bit for bit."""
import numpy as np
import pytest

from glslpt._capi import PT_MODE_PLAIN, PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for
from test_tile_entry import lights_in_view

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


@pytest.mark.parametrize("mode", [PT_MODE_PLAIN, PT_MODE_WAVEFRONT])
@pytest.mark.parametrize("width,height,fov,ratio", [(1920, 1080, 40.0, 1e-4), (1280, 720, 1.0, 3e-4), (1280, 720, 0.09, 1e-4)])
def test_ten_samples_at_once(renderer, mode, width, height, fov, ratio):
    sc, rs, cam, _ = lights_in_view(np.random.default_rng(9), 24, width, height, fov, ratio)
    renderer.upload_scene(sc)
    renderer.set_options(options_for(rs, mode=mode, wave_spp=10, hide_emitters=0))
    renderer.set_camera(cam)
    renderer.clear()
    renderer.render(0, 10)
    renderer.synchronize()
    got = renderer.read_accum()
    renderer.clear()
    for s in range(10):
        renderer.render(s, 1)
    renderer.synchronize()
    want = renderer.read_accum()
    assert want[..., :3].max() > 3.5  # a light is seen (the sky gives 3)
    assert np.array_equal(got, want)
