"""Passes in two parts where they meet: renderers on two streams at once (threads of their own), two renderers that share a
stream's buffers, and the engine's passes over the reference layout, whose images are those of the renderer's reference
traversal."""
import threading

import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

SPECS = [(521, 509, 8, 4, 7), (360, 365, 16, 3, 11)]  # width, height, samples, depth, seed: 2.1M paths a pass


def bits(a):
    return a.view(np.uint32)


def one_by_one(scene, spp, **o):
    r = gpr.Renderer(scene, **o)
    for _ in range(spp):
        r.render(1)
    a = r.read()[0]
    r.free()
    return a


def test_two_streams_at_once():
    import torch
    scenes = [gpr.Scene.sphere_grid(w, h, 4) for w, h, *_ in SPECS]
    want = [one_by_one(s, spp, max_depth=d, rr_start=2, seed=seed) for s, (_, _, spp, d, seed) in zip(scenes, SPECS)]
    streams = [torch.cuda.Stream() for _ in SPECS]
    got, errors = [[], []], []

    def work(k):
        try:
            _, _, spp, d, seed = SPECS[k]
            gpr.set_stream(streams[k].cuda_stream)
            r = gpr.Renderer(scenes[k], max_depth=d, rr_start=2, seed=seed)
            for _ in range(4):
                r.reset()
                r.render(spp)
                got[k].append(r.read()[0])
            r.free()
        except Exception as e:  # reported by the main thread
            errors.append(e)
        finally:
            gpr.set_stream(0)

    print("[parts] two streams", flush=True)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for k in range(2):
        assert len(got[k]) == 4
        for g in got[k]:
            assert np.array_equal(bits(g), bits(want[k]))
    for st in streams:
        gpr.release_stream(st.cuda_stream)


def test_two_renderers_share_a_stream():
    print("[parts] one stream", flush=True)
    scenes = [gpr.Scene.sphere_grid(w, h, 4) for w, h, *_ in SPECS]
    opts = [dict(max_depth=d, rr_start=2, seed=seed) for _, _, _, d, seed in SPECS]
    want = [one_by_one(s, spec[2], **o) for s, spec, o in zip(scenes, SPECS, opts)]
    rs = [gpr.Renderer(s, **o) for s, o in zip(scenes, opts)]
    for _ in range(2):  # the other one's pass was captured with smaller buffers
        for k in (1, 0, 1):
            rs[k].reset()
            rs[k].render(SPECS[k][2])
            assert np.array_equal(bits(rs[k].read()[0]), bits(want[k]))
    for r in rs:
        r.free()


@pytest.mark.parametrize("capacity", [1 << 19, 1 << 22])
def test_reference_layout_of_an_engine_pass(capacity):
    s = gpr.Scene.sphere_grid(8, 8, 4)
    c = gpr.lookat((0, 0, 0), (1.0, 6, 9))
    want = []
    for w, h, spp, d, seed in SPECS:
        s.set_camera(c, 40, w, h)
        want.append(one_by_one(s, spp, max_depth=d, rr_start=3, seed=seed, traversal=gpr.TRAVERSAL_REF))
    b = gpr.Batch(gpr.arena_bytes(s), capacity=capacity, max_jobs=4)
    i = b.add_scene(s)
    for w, h, spp, d, seed in SPECS:
        b.add_job(gpr.job(i, w, h, spp, c, 40, d, 3, seed))
    print(f"[parts] reference layout, capacity {capacity}", flush=True)
    b.set_cfg(256, 16, 64, 1, 0)
    for _ in range(2):
        b.run()
        for k, w in enumerate(want):
            assert np.array_equal(bits(b.read(k)), bits(w)), k
    b.free()
