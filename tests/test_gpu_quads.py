"""Short batches walk a ray with four lanes: hits have the bits of the one-lane walk that a chosen launch shape runs."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

QUAD_RAYS = 1 << 17  # the longest batch in this form


def rays(n, seed):
    g = np.random.default_rng(seed)
    r = np.zeros(n, gpr.RAY_DTYPE)
    f = r.view(np.float32).reshape(n, 8)
    f[:, 0:3] = g.random((n, 3))
    f[:, 3:6] = g.normal(size=(n, 3))
    f[:, 7] = np.inf
    k = np.arange(n)
    f[k % 7 == 1, 3] = 0.0                      # in a slab plane's direction
    f[k % 7 == 2, 3:5] = (0.0, -0.0)            # along an axis
    f[k % 7 == 3, 6:8] = (-0.5, 0.5)            # segments on both sides of the origin
    f[k % 7 == 4, 6:8] = (0.1, 0.2)
    f[k % 11 == 5, 0:3] *= 4                    # from outside
    f[k % 101 == 6, 3] = np.inf
    f[k % 101 == 7, 4] = np.nan
    f[k % 101 == 8, 3:6] = 0.0
    return r


def soup(n, seed):
    g = np.random.default_rng(seed)
    p = (g.random((n, 1, 3)) + 0.5 * n ** (-1 / 3) * g.normal(size=(n, 3, 3))).astype(np.float32)
    p[n // 2: n // 2 + n // 8] = p[0]           # equal triangles: equal keys, a deep tree, ties of t
    p[n // 4: n // 4 + n // 16, 2] = p[n // 4: n // 4 + n // 16, 1]  # without area
    return p.reshape(n, 9)


@pytest.mark.parametrize("ntri,n", [(1, 5), (2, 17), (3, 64), (5, 1), (70, 3), (3000, 4097), (3000, 65537), (60000, 16),
                                    (60000, QUAD_RAYS - 1), (60000, QUAD_RAYS), (60000, QUAD_RAYS + 1)])
@pytest.mark.parametrize("any_hit", [False, True])
def test_four_lanes_to_a_ray(ntri, n, any_hit):
    print(f"[quads] {ntri} triangles {n} rays any {any_hit}", flush=True)
    s = gpr.Scene.soup(soup(ntri, ntri)).commit()
    r = rays(n, n)
    got = s.trace(r, any_hit=any_hit)
    s.trace_set_cfg(128, 16, 64)
    want = s.trace(r, any_hit=any_hit)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s.free()


@pytest.mark.parametrize("name,w,h,spp", [("spheres", 256, 256, 4), ("textured", 257, 255, 3), ("spheres", 91, 90, 8), ("spheres", 181, 182, 8)])
def test_short_queues_of_a_render(name, w, h, spp):
    # one sample a pass keeps the queues below 2^17 entries (four lanes to an entry), all of them in one mostly exceed it
    import gpu_scenes as G
    s = gpr.Scene.sphere_grid(w, h, 6) if name == "spheres" else G.textured(w, h).commit()
    o = dict(max_depth=8, rr_start=3, seed=3)
    print(f"[quads] {name} {w}x{h} spp {spp}", flush=True)
    one, many = gpr.Renderer(s, **o), gpr.Renderer(s, **o)
    for _ in range(spp):
        one.render(1)
    many.render(spp)
    assert np.array_equal(one.read()[0].view(np.uint32), many.read()[0].view(np.uint32))
    one.free()
    many.free()


def test_short_queues_of_the_engine_against_refilled_walks():
    s = gpr.Scene.sphere_grid(8, 8, 6)
    b = gpr.Batch(gpr.arena_bytes(s), capacity=1 << 18, max_jobs=2)
    i = b.add_scene(s)
    for w, h in ((201, 77), (64, 33)):
        b.add_job(gpr.job(i, w, h, 3, gpr.lookat((0, 0, 0), (1.0, 6, 9)), 40, 6, 3, w))
    out = []
    for cfg in ((256, 16, 64, 0, 0), (64, 8, 64, 0, 0), (512, 8, 128, 0, 0), (128, 16, 64, 0, 1)):
        print(f"[quads] engine cfg {cfg}", flush=True)
        b.set_cfg(*cfg)
        b.run()
        out.append([b.read(0), b.read(1)])
    for o in out:
        assert all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(o, out[-1]))
    b.free()
