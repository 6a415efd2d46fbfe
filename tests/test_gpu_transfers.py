"""Ray queries and images that go through pinned memory in parts on several
host threads: sizes at the edges of the parts, against the oracle; several
handles at a time; arrays that share memory."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle
from common import oracle_setup, random_dirs, rel_err, small_instanced
from glslpt import _capi as api
from glslpt import scenes
from glslpt.renderer import Renderer, options_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def renderer():
    r = Renderer(0)
    yield r
    r.close()


def rays(n, seed=31):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-6, 6, (n, 3)).astype(np.float32), random_dirs(rng, n),
            rng.uniform(0.1, 10, n).astype(np.float32))


@pytest.fixture(scope="module")
def answers():
    """The oracle's for the largest size; smaller ones take its beginning."""
    sc, rs = small_instanced()
    sa, cam, o = oracle_setup(sc, rs)
    ro, rd, md = rays(262401)
    return oracle.closest_hit(sa, o, ro, rd), oracle.any_hit(sa, o, ro, rd, md)


def check(g, occ, want, n):
    ref, refocc = want
    same = (g["triangle"] == ref["triangle"][:n]) & (g["instance"] == ref["instance"][:n]) & (g["light"] == ref["light"][:n])
    # as the other query tests: ids of 0.9999 of the rays (one of a small set), t to 1e-5
    assert (~same).sum() <= max(1, n // 10000)
    both = same & (g["t"] < 1e6)
    assert rel_err(g["t"][both], ref["t"][:n][both]).max(initial=0.0) <= 1e-5
    assert (occ != refocc[:n]).sum() <= max(1, n // 10000)


@pytest.mark.parametrize("n", [1, 49, 255, 257, 32768, 32769, 65537, 98305, 131072, 131073, 262144, 262401])
@pytest.mark.parametrize("width", [2, 4])
def test_query_parts(renderer, answers, n, width):
    sc, rs = small_instanced()
    renderer.upload_scene(sc)
    renderer.set_options(options_for(rs, bvh_width=width))
    ro, rd, md = (a[:n] for a in rays(262401))
    check(renderer.closest_hit(ro, rd), renderer.any_hit(ro, rd, md), answers, n)


def test_query_arrays_that_share_memory(renderer):
    """Answers written over the inputs, and two answers to one array (the later
    one stays), over several parts."""
    sc, rs = small_instanced()
    renderer.upload_scene(sc)
    renderer.set_options(options_for(rs))
    n = 150001
    ro, rd, md = rays(n)
    want, occ = renderer.closest_hit(ro, rd), renderer.any_hit(ro, rd, md)
    o, d, uv = ro.copy(), rd.copy(), np.zeros((n, 2), np.float32)
    li = np.zeros(n, np.int32)
    t = o.reshape(-1)[:n]  # the front of the origins
    inst = d.reshape(-1)[n:2 * n].view(np.int32)
    lib, h = renderer._lib, renderer._h
    assert lib.pt_closest_hit(h, api.fptr(o), api.fptr(d), n, api.fptr(t), api.iptr(inst), uv.ctypes.data_as(C.POINTER(C.c_int32)),
                              api.iptr(li), api.fptr(uv)) == 0
    assert np.array_equal(t, want["t"]) and np.array_equal(inst, want["instance"])
    assert np.array_equal(li, want["light"]) and np.array_equal(uv, want["uv"])
    m = md.copy()
    assert lib.pt_any_hit(h, api.fptr(ro), api.fptr(rd), api.fptr(m), n, m.ctypes.data_as(C.POINTER(C.c_int32))) == 0
    assert np.array_equal(m.view(np.int32), occ)


@pytest.mark.parametrize("size", [(1, 1), (362, 362), (363, 363), (725, 725), (1031, 1021)])
def test_image_parts(renderer, size):
    """Float images of 16 bytes to 8 parts (2 MB is 362.04 squared pixels; 725
    squared the same for bytes) against the oracle's."""
    sc, rs = scenes.cornell()
    rs.width, rs.height, rs.max_depth = size[0], size[1], 1
    renderer.upload_scene(sc)
    sa, cam, o = oracle_setup(sc, rs)
    ref = oracle.render(sa, cam, o, 0, 1)
    renderer.set_options(options_for(rs))
    renderer.set_camera(sc.camera())
    renderer.clear()
    renderer.render(0, 1)
    got = renderer.read_accum()  # waits for the render by itself
    e = rel_err(got[..., :3], ref[..., :3], floor=1e-4).max(axis=2)
    assert (e <= 1e-4).mean() >= 0.999
    ldr = renderer.read_ldr(1).astype(np.int64)
    d = np.abs(ldr - oracle.tonemap(got, 1))
    assert d.max() <= 1 and (d > 0).mean() < 1e-3
    renderer.synchronize()


def test_several_handles_at_a_time(answers):
    """Six threads with a handle each, more lanes than are kept; the last handle
    gives them back and a later one makes them anew."""
    sc, rs = small_instanced()
    n = 200003
    ro, rd, md = (a[:n] for a in rays(262401))
    errors = []

    def work():
        try:
            r = Renderer(0)
            r.upload_scene(sc)
            r.set_options(options_for(rs))
            for _ in range(3):
                check(r.closest_hit(ro, rd), r.any_hit(ro, rd, md), answers, n)
            r.close()
        except BaseException as e:
            errors.append(e)

    for _ in range(2):
        ts = [threading.Thread(target=work) for _ in range(6)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not errors, errors


@pytest.mark.parametrize("graph", [0, 1])
def test_batch_images_that_share_memory(renderer, graph):
    """Two jobs with one output array: the later job's image stays."""
    sc, rs, jobs = scenes.batch_jobs(4)
    jobs = [dict(j, width=500 + 7 * i, height=401, spp=1, max_depth=2) for i, j in enumerate(jobs)]
    renderer.upload_scene(sc)
    renderer.set_options(options_for(rs, wave_spp=1, use_graph=graph))
    want = renderer.batch_render(jobs)
    assert all(w.any() for w in want)
    outs = [np.zeros_like(w) for w in want]
    arr = (api.PtJob * 4)()
    for i, j in enumerate(jobs):
        arr[i].camera, arr[i].width, arr[i].height = j["camera"], j["width"], j["height"]
        arr[i].spp, arr[i].max_depth = j["spp"], j["max_depth"]
        arr[i].accum_out = api.fptr(outs[2 if i == 1 else i])
    assert renderer._lib.pt_batch_render(renderer._h, arr, 4) == 0
    for i in (0, 2, 3):
        assert np.array_equal(outs[i], want[i])
