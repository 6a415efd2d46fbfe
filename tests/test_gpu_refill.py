"""Lanes that begin a new path while the rest of their wave goes on (k_finish and
the plain form in scenes of few triangles): images equal those of the staged
form (compact_every 2) bit for bit, at sizes around the waves' shares and at
sample counts around a launch's 16."""
import numpy as np
import pytest

from glslpt import scenes
from glslpt._capi import PT_MODE_PLAIN, PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for
from test_gpu_finish import image

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


@pytest.mark.parametrize("kind,size,spp", [
    ("media", (1, 1), 1), ("media", (1, 1), 33), ("media", (63, 65), 15), ("media", (200, 117), 17),
    ("textures", (1030, 515), 16), ("alpha_mask", (1030, 515), 3), ("volmis", (1030, 515), 2), ("volmis", (700, 515), 18),
    ("alpha_blend", (700, 515), 18)])
def test_refilled_lanes(renderer, kind, size, spp):
    """k_finish: 1 path to 6.6M (50 per lane), so waves take their first paths,
    parts of 8 to 64 and the last ones; volmis and alpha_blend: on both sides of
    16 paths per lane. Plain form: one launch, one of 16 samples and a rest."""
    sc, rs = scenes.feature_scene(kind, width=size[0], height=size[1], spp=spp, max_depth=6)
    renderer.upload_scene(sc)
    want = image(renderer, sc, rs, PT_MODE_WAVEFRONT, spp, wave_spp=spp, compact_every=2)
    renderer.reset_stats()
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, spp, wave_spp=spp)
    assert np.isfinite(want).all() and np.array_equal(got, want)
    assert np.array_equal(image(renderer, sc, rs, PT_MODE_PLAIN, spp), want)
