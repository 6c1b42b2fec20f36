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
