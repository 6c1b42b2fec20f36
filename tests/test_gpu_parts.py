"""Large passes run as two chains of launches side by side: images and queue sizes are those of passes in one part."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

SPLIT = 1 << 21        # paths from which a renderer's pass has two parts
ENGINE_SPLIT = 5 << 18  # the multi-job engine's


def bits(a):
    return a.view(np.uint32)


# at the size, just above (an odd remainder in the second part), just below, and one sample of a large image
@pytest.mark.parametrize("w,h,spp", [(512, 512, 8), (521, 509, 8), (512, 511, 8), (1531, 1401, 2)])
def test_parts_of_a_renderer_pass(w, h, spp):
    s = gpr.Scene.sphere_grid(w, h, 4)
    o = dict(max_depth=4, rr_start=2, seed=7)
    print(f"[parts] {w}x{h} spp {spp}", flush=True)
    one = gpr.Renderer(s, **o)
    for _ in range(spp):
        one.render(1)
    r = gpr.Renderer(s, **o)
    for _ in range(3):  # replays of the captured pass
        r.reset()
        r.render(spp)
        assert np.array_equal(bits(r.read()[0]), bits(one.read()[0]))
    assert all(np.array_equal(a, b) for a, b in zip(r.queue_sizes(4), one.queue_sizes(4)))
    ref = gpr.Renderer(s, traversal=gpr.TRAVERSAL_REF, **o)
    ref.render(spp)
    assert all(np.array_equal(a, b) for a, b in zip(r.queue_sizes(4), ref.queue_sizes(4)))
    for x in (one, r, ref):
        x.free()


@pytest.mark.parametrize("capacity", [ENGINE_SPLIT - 1, ENGINE_SPLIT, 1 << 22])
def test_parts_of_an_engine_pass(capacity):
    s = gpr.Scene.sphere_grid(8, 8, 4)
    specs = [(360, 365, 8, 3), (33, 17, 5, 6), (513, 511, 16, 2)]
    c = gpr.lookat((0, 0, 0), (1.0, 6, 9))
    want = []
    for w, h, spp, d in specs:
        s.set_camera(c, 40, w, h)
        r = gpr.Renderer(s, max_depth=d, rr_start=3, seed=w)
        for _ in range(spp):
            r.render(1)
        want.append(r.read()[0])
        r.free()
    b = gpr.Batch(gpr.arena_bytes(s), capacity=capacity, max_jobs=4)
    srv = gpr.Server(gpr.arena_bytes(s) + (4 << 30), gpr.arena_bytes(s), capacity=capacity, max_jobs=4)
    ib, isv = b.add_scene(s), srv.add_scene(s)
    jobs = [(w, h, spp, c, 40, d, 3, w) for w, h, spp, d in specs]
    for j in jobs:
        b.add_job(gpr.job(ib, *j))
    for cfg in ((256, 16, 64, 0, 0), (64, 8, 64, 0, 1), (256, 16, 64, 1, 0)):
        print(f"[parts] engine capacity {capacity} cfg {cfg}", flush=True)
        b.set_cfg(*cfg)
        b.run()
        for k, w in enumerate(want):
            if cfg[3] == 0:
                assert np.array_equal(bits(b.read(k)), bits(w)), k
    tickets = [srv.submit(gpr.job(isv, *j)) for j in jobs]
    for t, w in zip(tickets, want):
        assert np.array_equal(bits(srv.wait(t)[0]), bits(w))
    b.free()
    srv.free()
