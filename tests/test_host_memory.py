"""What the renderer's host code does with memory: calls where pinned memory
cannot be had. CPU build over a stand-in HIP runtime."""
import numpy as np
import pytest

import hostabi
from common import random_dirs, small_instanced
from glslpt.renderer import options_for


@pytest.fixture
def renderer():
    r = hostabi.HostRenderer()
    yield r
    hostabi.lib().fake_refuse_pinned(0)
    hostabi.lib().fake_device_limit(2 ** 64 - 1)
    r.close()
    assert hostabi.lib().fake_device_used() == 0 and hostabi.lib().fake_pinned() == 0


def scene(r, **opts):
    sc, rs = small_instanced()
    r.upload_scene(sc)
    r.set_options(options_for(rs, **opts))
    r.set_camera(sc.camera())
    return sc, rs


@pytest.mark.parametrize("n", [1, 255, 257, 65537, 131073])
def test_queries_without_pinned_memory(renderer, n):
    scene(renderer)
    rng = np.random.default_rng(1)
    ro = rng.uniform(-6, 6, (n, 3)).astype(np.float32)
    rd, md = random_dirs(rng, n), rng.uniform(0.1, 10, n).astype(np.float32)
    want, occ = renderer.closest_hit(ro, rd), renderer.any_hit(ro, rd, md)
    assert n < 100 or (0 < occ.sum() < n and (want["triangle"] >= 0).any())
    renderer.close()  # the lanes go with the last renderer
    renderer.__init__()
    hostabi.lib().fake_refuse_pinned(1)
    scene(renderer)
    got, gocc = renderer.closest_hit(ro, rd), renderer.any_hit(ro, rd, md)
    for k in want:
        assert np.array_equal(got[k], want[k])
    assert np.array_equal(gocc, occ)


def test_renders_without_pinned_memory(renderer):
    hostabi.lib().fake_refuse_pinned(1)
    sc, rs = scene(renderer)
    renderer.clear()
    renderer.render(0, 2)
    renderer.synchronize()
    assert renderer.read_accum().shape == (rs.height, rs.width, 4)
    assert renderer.stats()["stack_overflow"] == 0
    job = dict(camera=sc.camera(), width=20, height=10, spp=2, max_depth=3)
    assert renderer.batch_render([job])[0].shape == (10, 20, 4)
    renderer.adjoint(0, 1, np.zeros((rs.height, rs.width, 3), np.float32))
