"""Materials that start to blend, or cease to, in an instance edit: the image is
that of a fresh upload of the same scene, bit for bit, in every form."""
import ctypes as C

import numpy as np
import pytest

from glslpt import _capi as api
from glslpt import scenes
from glslpt._capi import PT_MODE_PLAIN, PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for
from test_gpu_finish import image

pytestmark = pytest.mark.gpu
ALPHA_MODE = 29  # floats of a material: opacity, alphaMode, alphaCutoff at 28..30


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


def table(sc, mode):
    """The scene's materials with every alpha-tested one set to `mode`."""
    v = sc.view()
    m = np.ctypeslib.as_array(C.cast(v.materials, C.POINTER(C.c_float)), (v.num_materials, 32)).copy()
    tested = m[:, ALPHA_MODE] != 0
    assert tested.any()
    m[tested, ALPHA_MODE] = mode
    m[tested, ALPHA_MODE - 1] = 0.45
    return m


@pytest.mark.parametrize("width", [2, 4])
@pytest.mark.parametrize("mode", [PT_MODE_PLAIN, PT_MODE_WAVEFRONT])
@pytest.mark.parametrize("before,after", [(2, 1), (1, 2)])
def test_blending_follows_the_table(renderer, mode, width, before, after):
    sc, rs = scenes.feature_scene("alpha_mask", width=120, height=80, spp=4, max_depth=5)
    opts = dict(bvh_width=width, wave_spp=4)
    job = [dict(camera=sc.camera(), width=90, height=70, spp=3, max_depth=4)]
    renderer.upload_scene(sc, materials=table(sc, after))
    want = image(renderer, sc, rs, mode, 4, **opts), renderer.batch_render(job)[0]
    renderer.upload_scene(sc, materials=table(sc, before))
    first = image(renderer, sc, rs, mode, 4, **opts)
    v, m = sc.view(), table(sc, after)
    renderer._check("pt_update_instances", renderer._lib.pt_update_instances(
        renderer._h, v.transforms, v.num_instances, C.cast(m.ctypes.data, C.POINTER(api.PtMaterial)),
        v.num_materials, None, 0, 0))
    got = image(renderer, sc, rs, mode, 4, **opts), renderer.batch_render(job)[0]
    assert not np.array_equal(first, want[0])
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
