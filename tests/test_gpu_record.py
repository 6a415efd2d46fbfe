"""The adjoint's recorded hits: the replay takes the closest hits of its
first bounces from the primal pass, whether its stages or the launch that runs
paths to their end (k_finish) found them, and queries later ones again."""
import numpy as np
import pytest

from common import oracle_setup
from glslpt import scenes
from glslpt.renderer import Renderer, options_for
from test_gpu_adjoint import _compare_frozen, frozen_fd, small_boxes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


def adjoint(r, sc, rs, w, spp, **kw):
    r.set_options(options_for(rs, **kw))
    r.set_camera(sc.camera())
    g = r.adjoint(0, spp, w).astype(np.float64)
    assert r.stats()["adjoint_dropped"] == 0
    return g


@pytest.mark.parametrize("cadence", [1, 2])
@pytest.mark.parametrize("depth", [0, 15, 16, 24])
def test_depths_around_the_record(renderer, depth, cadence):
    """depth + 1 bounces without Russian roulette against the oracle's frozen
    differences, with the tolerance of the other comparisons with it."""
    sc, rs = small_boxes(num_materials=6, width=32, height=32)
    rs.max_depth, rs.enable_rr = depth, False
    renderer.upload_scene(sc)
    sa, cam, o = oracle_setup(sc, rs)
    w = np.random.default_rng(61).normal(size=(rs.height, rs.width, 3)).astype(np.float32)
    g = adjoint(renderer, sc, rs, w, rs.spp, wave_spp=4, compact_every=cadence)
    pick = [(m, k) for m in range(sa.a["materials"].shape[0]) for k in (0, 1, 2)]
    fd = frozen_fd(sa, cam, o, w, rs.spp, pick)
    got = np.array([g[m, k] for m, k in pick])
    if not fd.any():  # depth 0: emitted light alone, which these parameters do not change
        assert not got.any()
        return
    _, rel = _compare_frozen(f"depth {depth}", got, fd, pick)
    assert rel.max() <= 0.01


@pytest.mark.parametrize("size,spp,depth", [((1, 1), 3, 4), ((63, 65), 5, 4), ((512, 512), 16, 4), ((512, 512), 16, 24)])
@pytest.mark.parametrize("cadence", [1, 2])
def test_one_pass_equals_many(renderer, size, spp, depth, cadence):
    """25 bounces of 4.2M paths are more than the record's 2 GB hold (16), those
    of one sample are not. 4.2M paths in one pass are staged and their tail finished in one launch;
    one sample per pass runs whole (compact_every 2: staged). The sums differ by
    rounding alone: 1e-4 of the largest entry, for partial sums of ~1e4 terms in
    fp32 (1e4^0.5 * 6e-8) with tenfold cancellation."""
    sc, rs = scenes.material_boxes(width=size[0], height=size[1], max_depth=depth)
    rs.enable_rr = depth < 24
    renderer.upload_scene(sc)
    w = np.random.default_rng(62).normal(size=(rs.height, rs.width, 3)).astype(np.float32)
    a = adjoint(renderer, sc, rs, w, spp, wave_spp=spp, compact_every=cadence)
    b = adjoint(renderer, sc, rs, w, spp, wave_spp=1)
    assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max()
