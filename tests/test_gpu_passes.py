"""Passes of several samples on the GPU: an image rendered in passes of many samples has the bits of the same samples
rendered one at a time, and the reported queue sizes are those of the last sample."""
import threading

import numpy as np
import pytest

import gpr
import gpu_scenes as G

pytestmark = pytest.mark.gpu


def scene(name, w, h):
    if name == "cornell":
        return gpr.Scene.cornell(w, h)
    if name == "spheres":
        return gpr.Scene.sphere_grid(w, h, 6)
    return G.textured(w, h).commit()


def by_ones(s, spp, **o):
    r = gpr.Renderer(s, **o)
    for _ in range(spp):
        r.render(1)
    out = r.read(), r.queue_sizes(o["max_depth"])
    r.free()
    return out


@pytest.mark.parametrize("name,w,h,spp,depth", [
    ("cornell", 1, 1, 64, 5), ("cornell", 63, 9, 7, 3), ("cornell", 33, 31, 128, 1), ("spheres", 65, 17, 13, 8),
    ("spheres", 7, 130, 21, 64), ("textured", 40, 33, 16, 6), ("cornell", 16, 8, 5, 0)])
@pytest.mark.parametrize("traversal", [gpr.TRAVERSAL_FAST, gpr.TRAVERSAL_REF])
def test_many_samples_a_pass_equal_one(name, w, h, spp, depth, traversal):
    s = scene(name, w, h)
    o = dict(max_depth=depth, rr_start=2, seed=11, traversal=traversal)
    print(f"[passes] {name} {w}x{h} spp {spp} depth {depth}", flush=True)
    (want, wcnt), (wsh, wsc) = by_ones(s, spp, **o)
    r = gpr.Renderer(s, **o)
    r.render(spp)
    got, cnt = r.read()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(cnt, wcnt)
    sh, sc = r.queue_sizes(depth)
    # 2^k samples leave a last pass of many samples, other counts one of a single sample
    assert np.array_equal(sh, wsh) and np.array_equal(sc, wsc)
    # progressive calls split the passes differently
    r.reset()
    for part in (spp // 3, spp - spp // 3):
        r.render(part)
    again, _ = r.read()
    assert np.array_equal(again.view(np.uint32), want.view(np.uint32))
    r.free()


def test_renderers_of_one_stream_share_the_pass_buffers():
    # a small shallow image, a larger one, a deeper one, then the first again: the buffers grow between its passes
    specs = [("cornell", 24, 24, 3), ("spheres", 90, 70, 4), ("cornell", 24, 24, 9)]
    scenes = [scene(n, w, h) for n, w, h, _ in specs]
    opts = [dict(max_depth=d, rr_start=3, seed=5) for _, _, _, d in specs]
    want = [by_ones(s, 24, **o)[0][0] for s, o in zip(scenes, opts)]
    rs = [gpr.Renderer(s, **o) for s, o in zip(scenes, opts)]
    for part in (8, 16):
        for r in rs:
            r.render(part)
    for r, w in zip(rs, want):
        assert np.array_equal(r.read()[0].view(np.uint32), w.view(np.uint32))
    # the same from two threads on the one stream
    for r in rs:
        r.reset()
    ts = [threading.Thread(target=r.render, args=(24,)) for r in rs]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for r, w in zip(rs, want):
        assert np.array_equal(r.read()[0].view(np.uint32), w.view(np.uint32))
        r.free()


def test_options_and_camera_change_between_passes():
    s = scene("spheres", 48, 40)
    r = gpr.Renderer(s, max_depth=3, seed=1)
    r.render(8)
    for depth, mode in ((9, gpr.RNG_PCG), (4, gpr.RNG_REFERENCE), (2, gpr.RNG_PCG)):
        r.set_opts(max_depth=depth, seed=3, rng_mode=mode)
        s.set_camera_lookat((0, 0, 0), (depth * 0.1, 6, 10), (0, 1, 0), 40, 48, 40)
        r.render(10)
        got = r.read()[0]
        want = by_ones(s, 10, max_depth=depth, seed=3, rng_mode=mode)[0][0]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (depth, mode)
    r.free()


@pytest.mark.parametrize("capacity", [1500, 5000, 1 << 16, 1 << 20])
def test_jobs_with_uneven_samples(capacity):
    # jobs run out of samples at different passes; the capacity decides how many samples a pass holds
    s = scene("spheres", 8, 8)
    specs = [(37, 40, 1, 5), (9, 8, 64, 64), (33, 17, 5, 2), (1, 1, 130, 3), (20, 20, 16, 8)]
    cams = [gpr.lookat((0, 0, 0), (1.0 + k, 6, 9)) for k in range(len(specs))]
    b = gpr.Batch(gpr.arena_bytes(s), capacity=capacity, max_jobs=8)
    srv = gpr.Server(gpr.arena_bytes(s) + (1 << 30), gpr.arena_bytes(s), capacity=capacity, max_jobs=8)
    ib, isv = b.add_scene(s), srv.add_scene(s)
    jobs = [(w, h, spp, c, 40, d, 3, 21 + w) for (w, h, spp, d), c in zip(specs, cams)]
    for j in jobs:
        b.add_job(gpr.job(ib, *j))
    b.run()
    tickets = [srv.submit(gpr.job(isv, *j)) for j in jobs]
    served = [srv.wait(t)[0] for t in tickets]
    for k, ((w, h, spp, d), c) in enumerate(zip(specs, cams)):
        s.set_camera(c, 40, w, h)
        want = by_ones(s, spp, max_depth=d, rr_start=3, seed=21 + w)[0][0]
        assert np.array_equal(b.read(k).view(np.uint32), want.view(np.uint32)), k
        assert np.array_equal(served[k].view(np.uint32), want.view(np.uint32)), k
    b.run()  # again from the first sample
    assert np.array_equal(b.read(0).view(np.uint32), served[0].view(np.uint32))
    assert b.stats().paths == sum(w * h * spp for w, h, spp, _ in specs)
    b.free()
    srv.free()


@pytest.mark.parametrize("rng_mode", [gpr.RNG_REFERENCE, gpr.RNG_PCG])
@pytest.mark.parametrize("depth", [4, 5, 6, 12])
def test_terms_of_paths_that_end_at_a_light(rng_mode, depth):
    # a grey floor under a grey light the size of the floor, and a sky: scattered rays meet the light at every bounce,
    # the last one included, and in reference RNG mode the roulette turns some of those hits into misses of the sky
    from test_gpu_render import gpu_render, oracle_render
    s = gpr.Scene()
    for y, e in ((-1.0, 0.0), (1.0, 2.0)):
        p, uv, c = G._quad([(-3, y, -3), (3, y, -3), (3, y, 3), (-3, y, 3)], [(0, 0), (1, 0), (1, 1), (0, 1)])
        s.add_mesh(p if y < 0 else p[::-1].copy(), corners=c, uv=uv,
                   mat=gpr.material(gpr.MAT_DIFFUSE, color=(0.6, 0.5, 0.7), emission=(e, e, e)))
    s.set_env_map(s.add_texture(np.random.default_rng(1).random((8, 16, 3))), np.eye(4, dtype=np.float32))
    s.set_camera_lookat((0, 0, 0), (0.5, 0.2, 4.0), (0, 1, 0), 60, 37, 19)
    s.commit()
    print(f"[passes] light terms depth {depth} rng {rng_mode}", flush=True)
    for traversal in (gpr.TRAVERSAL_REF, gpr.TRAVERSAL_FAST):
        got, cnt, _, _ = gpu_render(s, 5, depth, rng_mode, 3, traversal)
        want, wcnt = oracle_render(s, 5, depth, rng_mode, 3)
        assert np.array_equal(cnt, wcnt)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s.free()
