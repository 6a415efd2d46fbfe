"""What the renderer's host code does with memory: calls where pinned memory or the
adjoint's record cannot be had. CPU build over a stand-in HIP runtime."""
import os
import subprocess
import sys

import numpy as np
import pytest

import hostabi
from common import random_dirs, small_instanced
from glslpt._capi import PtError
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


def adjoint_call(r, size, depth):
    sc, rs = small_instanced()
    rs.width = rs.height = size
    rs.max_depth = depth
    r.upload_scene(sc)
    r.set_options(options_for(rs, wave_spp=1, compact_every=2))
    r.set_camera(sc.camera())
    r.adjoint(0, 1, np.zeros((size, size, 3), np.float32))


SIDE = 2400  # 5.8M paths: 184 MB of record per bounce
EACH = 28 * (SIDE * SIDE + SIDE * SIDE // 7 + 64)


def test_record_kept_between_calls_is_bounded(renderer):
    """16 recorded bounces of 5.8M paths are 2.9 GB; at most 2 GB of them stay."""
    lib = hostabi.lib()
    adjoint_call(renderer, SIDE, 0)
    one = lib.fake_device_used()
    lib.fake_device_peak()
    adjoint_call(renderer, SIDE, 15)
    assert lib.fake_device_peak() - one > 14 * EACH * 0.85
    assert lib.fake_device_used() - one <= (2 << 30)


def test_record_of_fewer_bounces(renderer):
    """Where 16 bounces cannot be had but 6 can, some are recorded, and a call
    that needs the room gets it from the record."""
    lib = hostabi.lib()
    adjoint_call(renderer, SIDE, 0)
    one = lib.fake_device_used()
    limit = one + 6 * EACH
    lib.fake_device_limit(limit)
    lib.fake_device_peak()
    adjoint_call(renderer, SIDE, 15)
    assert lib.fake_device_peak() - one > 2 * EACH * 0.85
    kept = lib.fake_device_used()
    assert kept > one + EACH
    # a scene whose textures take all but what the record holds
    texels = (limit - kept) // 4 + (1 << 20)
    sc, rs = small_instanced()
    v = sc.view()
    tex = np.zeros(4 * texels, np.uint8)
    v.num_textures, v.tex_width, v.tex_height = 1, 1 << 10, (texels >> 10) - 1
    v.texture_maps = tex.ctypes.data_as(type(v.texture_maps))
    renderer._check("pt_upload_scene", lib.pt_upload_scene(renderer._h, hostabi.C.byref(v)))


@pytest.mark.parametrize("kind", ["whole", "staged", "counted", "batch", "batch staged", "adjoint", "adjoint staged"])
def test_depth_takes_little_memory(renderer, kind):
    """The counters of a pass are not held for every bounce that a depth allows
    (paths end by Russian roulette long before)."""
    lib = hostabi.lib()
    used = []
    for depth in (8, 20000):
        sc, rs = small_instanced()
        rs.max_depth = depth
        renderer.upload_scene(sc)
        renderer.set_options(options_for(rs, compact_every=2 if "staged" in kind else 1, count_work=kind == "counted"))
        renderer.set_camera(sc.camera())
        lib.fake_device_peak()
        if "batch" in kind:
            renderer.batch_render([dict(camera=sc.camera(), width=64, height=64, spp=2, max_depth=depth)])
        elif "adjoint" in kind:
            if depth > 8:  # the record and the visibility words, 28 bytes and two bits per path and bounce, aside
                rs.width = rs.height = 1
                renderer.set_options(options_for(rs, compact_every=2 if "staged" in kind else 1, wave_spp=1))
            renderer.adjoint(0, 1, np.zeros((rs.height, rs.width, 3), np.float32))
        else:
            renderer.clear()
            renderer.render(0, 2)
            renderer.synchronize()
        used.append(lib.fake_device_peak())
    room = 28 * 150 * 20000 + 128 * 20001 if "adjoint" in kind else 0
    assert used[1] - used[0] < (2 << 20) + room


@pytest.mark.parametrize("mode", [0, 1])
def test_small_batches_pin_little(renderer, mode):
    """What a lane pins follows the largest part that the call copies."""
    sc, rs = scene(renderer, mode=mode)
    jobs = [dict(camera=sc.camera(), width=40 + k, height=64, spp=1, max_depth=2) for k in range(6)]
    renderer.batch_render(jobs)
    assert hostabi.lib().fake_pinned() <= 6 * (64 << 10) + 64
    renderer.batch_render([dict(jobs[0], width=500, height=600)])
    assert hostabi.lib().fake_pinned() <= 9 * (4 << 20)


CALLS = {
    "upload": lambda r, sc, rs, q: r.upload_scene(sc),
    "closest 49": lambda r, sc, rs, q: r.closest_hit(q[0][:49], q[1][:49]),
    "closest 140000": lambda r, sc, rs, q: r.closest_hit(*q[:2]),
    "any 140000": lambda r, sc, rs, q: r.any_hit(*q),
    "render": lambda r, sc, rs, q: (r.render(0, 2), r.synchronize()),
    "image": lambda r, sc, rs, q: r.read_accum(),
    "batch": lambda r, sc, rs, q: r.batch_render(
        [dict(camera=sc.camera(), width=600 + k, height=500, spp=2, max_depth=3) for k in range(3)]),
    "adjoint": lambda r, sc, rs, q: r.adjoint(0, 1, np.zeros((rs.height, rs.width, 3), np.float32)),
}


def sweep(name):
    """Every host allocation of a call fails once: the call reports it, or does
    without, and the next one runs."""
    lib = hostabi.lib()
    lib.fake_fail_new.argtypes = [hostabi.C.c_long]
    lib.fake_fail_new.restype = None
    lib.fake_fail_new_left.restype = hostabi.C.c_long
    rng = np.random.default_rng(1)
    n = 140000
    q = (rng.uniform(-6, 6, (n, 3)).astype(np.float32), random_dirs(rng, n), np.ones(n, np.float32))
    r = hostabi.HostRenderer()
    sc, rs = scene(r)
    rs.width, rs.height = 700, 640  # an image of several parts
    r.set_options(options_for(rs))
    r.clear()
    failed = 0
    for k in range(100000):
        lib.fake_fail_new(k)
        try:
            CALLS[name](r, sc, rs, q)
        except PtError:
            failed += 1
        left = lib.fake_fail_new_left()
        lib.fake_fail_new(-1)
        if k % 7 == 0:
            CALLS[name](r, sc, rs, q)
        if left >= 0:  # the call made fewer allocations
            break
        if k % 5 == 4:  # again without idle lanes
            r.close()
            r.__init__()
            scene(r)
            r.set_options(options_for(rs))
            r.clear()
    r.close()
    assert lib.fake_device_used() == 0 and lib.fake_pinned() == 0
    print(f"{k} allocations, {failed} calls failed")


@pytest.mark.parametrize("name", CALLS)
def test_host_allocations_that_fail(name):
    """In a process of its own: a call that cannot handle it ends the process."""
    code = f"import test_host_memory as t; t.sweep({name!r})"
    env = dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path))
    p = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=600)
    print(p.stdout)
    assert p.returncode == 0, p.stderr[-2000:]
