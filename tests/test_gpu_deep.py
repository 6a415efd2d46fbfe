"""Deep passes in a closed room without Russian roulette, where paths go on to
the last bounce: passes that use their counters several times over, and the
takeover by k_finish after 40 bounces with more paths than its grid, give the
plain form's image bit for bit."""
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


def closed_room(width, height, spp, depth, spheres=20, freq=16):
    """Spheres in a box around the camera, everything diffuse and dimly glowing;
    20 spheres are 100k triangles over all instances."""
    rng = np.random.default_rng(17)
    sc = scenes.Scene()
    box = sc.AddMesh(*scenes._unit_box(), name="box")
    ball = sc.AddMesh(*scenes.displaced_icosphere(freq, 0.1, 5), name="sphere")
    mats = [sc.AddMaterial(baseColor=tuple(rng.uniform(0.9, 0.98, 3)), roughness=1.0,
                           emission=tuple(rng.uniform(0.01, 0.05, 3))) for _ in range(4)]
    sc.AddMeshInstance(box, scenes.mat4(scale=(20, 20, 20)), mats[0])
    for k in range(spheres):
        sc.AddMeshInstance(ball, scenes.mat4(translate=rng.uniform(-7, 7, 3)), mats[k % 4])
    sc.AddCamera((0.0, 0.0, 8.5), (0.0, 0.0, 0.0), 60.0)
    sc.ProcessScene()
    return sc, scenes.RenderSettings(width, height, spp, depth, enable_rr=False)


@pytest.mark.parametrize("depth", [254, 255, 256, 520])
def test_counters_used_again(renderer, depth):
    sc, rs = closed_room(40, 24, 3, depth, spheres=3, freq=4)
    renderer.upload_scene(sc)
    want = image(renderer, sc, rs, PT_MODE_PLAIN, 3)
    assert np.isfinite(want).all() and np.median(want[..., :3]) > 3 * 0.05 * 5  # light gathered over many bounces
    for cadence in (1, 2, 64):
        for opts in (dict(), dict(extend_cap=8), dict(nee_inline=1)):
            got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 3, wave_spp=3, compact_every=cadence, **opts)
            assert np.array_equal(got, want), (cadence, opts)
    hits = []
    for cadence in (1, 2):
        renderer.reset_stats()
        got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, 3, wave_spp=3, compact_every=cadence, count_work=1)
        assert np.array_equal(got, want)
        st = renderer.stats()
        hits.append(list(st["bounce_hits"]))
        assert sum(hits[-1]) <= st["rays_closest"] <= sum(hits[-1]) + 40 * 24 * 3
    assert hits[0] == hits[1] and hits[0][15] > 20 * 40 * 24 * 3


@pytest.mark.parametrize("graph", [0, 1])
def test_counters_used_again_in_a_batch(renderer, graph):
    sc, rs = closed_room(40, 24, 3, 300, spheres=3, freq=4)
    renderer.upload_scene(sc)
    jobs = [dict(camera=sc.camera(), width=33 + k, height=20, spp=2 + k, max_depth=d) for k, d in enumerate((300, 20, 257))]
    renderer.set_options(options_for(rs, mode=PT_MODE_PLAIN))
    want = renderer.batch_render(jobs)
    for cadence in (1, 2):
        renderer.set_options(options_for(rs, mode=PT_MODE_WAVEFRONT, wave_spp=2, use_graph=graph, compact_every=cadence))
        for got, w in zip(renderer.batch_render(jobs), want):
            assert np.array_equal(got, w)


def test_counters_used_again_in_the_adjoint(renderer):
    """The sums are of the same terms in another order."""
    sc, rs = closed_room(24, 16, 2, 300, spheres=3, freq=4)
    renderer.upload_scene(sc)
    dl = np.random.default_rng(5).normal(size=(16, 24, 3)).astype(np.float32)
    g = []
    for cadence in (1, 2, 64):
        renderer.set_options(options_for(rs, wave_spp=2, compact_every=cadence))
        renderer.set_camera(sc.camera())
        g.append(renderer.adjoint(0, 2, dl).astype(np.float64))
    assert np.abs(g[0]).max() > 0
    for other in g[1:]:
        # 2e5 terms per sum in fp32: 2e5^0.5 * 6e-8 with threefold cancellation
        assert np.abs(g[0] - other).max() <= 1e-4 * np.abs(g[0]).max()


@pytest.mark.parametrize("depth", [39, 40, 45, 60])
@pytest.mark.parametrize("kind", ["frame", "batch", "adjoint"])
def test_takeover_of_many_paths(renderer, kind, depth):
    """3.1M paths in a pass, staged up to bounce 40 (nearly all of them alive
    there, many times what the grid of k_finish holds at once) and taken over then."""
    size, spp = (1200, 864), 3
    sc, rs = closed_room(*size, spp, depth)
    renderer.upload_scene(sc)
    if kind == "adjoint":
        dl = np.random.default_rng(5).normal(size=(size[1], size[0], 3)).astype(np.float32)
        g = []
        for cadence in (1, 2):
            renderer.set_options(options_for(rs, wave_spp=spp, compact_every=cadence))
            renderer.set_camera(sc.camera())
            g.append(renderer.adjoint(0, spp, dl).astype(np.float64))
        assert np.abs(g[0]).max() > 0
        # up to 1e8 terms per sum in fp32, summed per block first: 1e4 of them in
        # a row at most, 1e4 * 6e-8 if their roundings all agreed
        assert np.abs(g[0] - g[1]).max() <= 6e-4 * np.abs(g[1]).max()
        return
    jobs = [dict(camera=sc.camera(), width=size[0], height=size[1], spp=spp, max_depth=depth)]
    if kind == "frame":
        want = image(renderer, sc, rs, PT_MODE_PLAIN, spp)
    else:
        renderer.set_options(options_for(rs, mode=PT_MODE_PLAIN))
        want, = renderer.batch_render(jobs)
    for cadence in (1, 2):
        if kind == "frame":
            renderer.reset_stats()
            got = image(renderer, sc, rs, PT_MODE_WAVEFRONT, spp, wave_spp=spp, compact_every=cadence)
            assert renderer.stats()["ms_stage"]["extend"] > 0
        else:
            renderer.set_options(options_for(rs, mode=PT_MODE_WAVEFRONT, wave_spp=spp, compact_every=cadence,
                                             use_graph=cadence - 1))
            got, = renderer.batch_render(jobs)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("cadence", [1, 2])
@pytest.mark.parametrize("depth", [15, 16, 24])
def test_record_boundary(renderer, depth, cadence):
    """The adjoint's record holds 16 bounces of 5.2M paths (2 GB hold 12) and all
    bounces of a sixth of them: queried again beyond bounce 15 or recorded, the
    gradient is the same up to the order of the sums (tolerance as above). A
    seventh of the light and more comes from the bounces beyond at depth 24."""
    size, spp = (1200, 864), 5
    sc, rs = closed_room(*size, spp, depth)
    renderer.upload_scene(sc)
    dl = np.random.default_rng(6).normal(size=(size[1], size[0], 3)).astype(np.float32)
    g = []
    for wave_spp in (5, 1):
        renderer.set_options(options_for(rs, wave_spp=wave_spp, compact_every=cadence))
        renderer.set_camera(sc.camera())
        g.append(renderer.adjoint(0, spp, dl).astype(np.float64))
    assert np.abs(g[1]).max() > 0
    assert np.abs(g[0] - g[1]).max() <= 6e-4 * np.abs(g[1]).max()
