"""k_finish's claims from several counters: passes of sizes around the first
batches that are dealt out so (2048 waves: 131072 paths at the start, 262144 at
the end), in views of next to nothing and of a room, equal the staged pass
(compact_every 2) bit for bit."""
import numpy as np
import pytest

from glslpt import scenes
from glslpt._capi import PT_MODE_WAVEFRONT
from glslpt.renderer import Renderer, options_for
from test_gpu_finish import image

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


@pytest.mark.parametrize("size,spp", [((8, 49152), 1), ((8, 49160), 1), ((8, 49208), 1), ((8, 49216), 1), ((8, 49224), 1),
                                      ((520, 256), 3), ((1021, 1031), 4)])
@pytest.mark.parametrize("kind", ["sky", "room", "volmis"])
def test_claims(renderer, kind, size, spp):
    if kind == "sky":
        sc, rs = scenes.instanced_spheres(num_instances=1, freq=4, width=size[0], height=size[1], max_depth=3)
        sc.AddCamera((0.0, 10.0, 60.0), (0.0, 0.0, 0.0), 100.0)
    else:
        sc, rs = scenes.feature_scene("media" if kind == "room" else kind, width=size[0], height=size[1], max_depth=4)
    renderer.upload_scene(sc)
    want = image(renderer, sc, rs, PT_MODE_WAVEFRONT, spp, wave_spp=spp, compact_every=2)
    renderer.reset_stats()
    got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, spp, wave_spp=spp)
    assert renderer.stats()["ms_stage"]["extend"] == 0  # run whole
    assert np.isfinite(want).all() and np.array_equal(got, want)
    jobs = [dict(camera=sc.camera(), width=size[0], height=size[1], spp=spp, max_depth=2)]
    out = []
    for cadence in (1, 2):
        renderer.set_options(options_for(rs, mode=PT_MODE_WAVEFRONT, wave_spp=spp, compact_every=cadence))
        out.append(renderer.batch_render(jobs)[0])
    assert np.array_equal(*out)
