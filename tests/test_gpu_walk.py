"""The BVH4 walk at the edges of its stack and of its key order on the GPU: walks deeper than the LDS part of the
stack, rays whose whole range lies behind their origin, and every launch shape giving the same hits."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

SHAPES = [(64, 8, 64, 0), (128, 8, 64, 1), (256, 16, 64, 0), (512, 32, 128, 1)]


def rays_between(o, p, tmin, tmax):
    r = np.zeros(len(o), gpr.RAY_DTYPE)
    r["o"], r["d"], r["tmin"], r["tmax"] = o, p - o, tmin, tmax
    return r


@pytest.mark.parametrize("ntri", [1, 2, 3, 5, 700, 20000])
@pytest.mark.parametrize("any_hit", [False, True])
def test_overlapping_boxes_fill_the_stack(ntri, any_hit):
    # thin triangles across the whole cube: nearly every box is entered, so walks push three children a node
    rng = np.random.default_rng(ntri)
    c = rng.random((ntri, 1, 3)).astype(np.float32)
    pos = (c + rng.normal(0, 0.4, (ntri, 3, 3))).astype(np.float32).reshape(ntri, 9)
    pos[:, 3:6] = pos[:, 0:3] + rng.normal(0, 1e-3, (ntri, 3)).astype(np.float32)
    s = gpr.Scene.soup(pos).commit()
    o, p = rng.random((2, 3000, 3)).astype(np.float32)
    r = rays_between(o, p, 0.0, 0.9999 if any_hit else np.inf)
    print(f"[walk] {ntri} slivers any={any_hit}", flush=True)
    ref = s.trace(r, any_hit=any_hit, ref_order=True)
    first = None
    for shape in SHAPES:
        s.trace_set_cfg(*shape)
        h = s.trace(r, any_hit=any_hit)
        first = h if first is None else first
        assert np.array_equal(h.view(np.uint32), first.view(np.uint32)), shape
    if any_hit:
        assert np.array_equal(first["id"] >= 0, ref["id"] >= 0)
    else:
        assert np.array_equal(first["id"], ref["id"])
        assert np.array_equal(first["t"].view(np.uint32), ref["t"].view(np.uint32))
    s.free()


@pytest.mark.parametrize("tmin,tmax", [(-2.0, -0.25), (-1.5, 0.5), (-np.inf, -0.1), (0.0, 0.0)])
def test_ranges_behind_the_origin(tmin, tmax):
    # entry distances are negative there: they order as 0 and must not be culled against a negative limit
    pos = gpr.gen_soup(3, 0, 5000, 0.03)
    s = gpr.Scene.soup(pos).commit()
    rng = np.random.default_rng(8)
    o, p = rng.random((2, 4000, 3)).astype(np.float32)
    r = rays_between(o, p, tmin, tmax)
    ref = s.trace(r, ref_order=True)
    for shape in SHAPES:
        s.trace_set_cfg(*shape)
        h = s.trace(r)
        assert np.array_equal(h["id"], ref["id"]), shape
    s.free()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4095, 4097, 8193, 40960, 40961, 131072, 131073, 200001])
def test_batch_sizes_around_the_spreading_of_short_batches(n):
    # short batches use thin waves; every ray is traced once whatever the share of a wave
    pos = gpr.gen_soup(5, 0, 3000, 0.03)
    s = gpr.Scene.soup(pos).commit()
    r = gpr.gen_rays(4, 1, n)
    for any_hit in (False, True):
        ref = s.trace(r, any_hit=any_hit, ref_order=True)
        for shape in SHAPES + [(256, 8, 192, 0), (256, 8, 192, 1)]:
            s.trace_set_cfg(*shape)
            h = s.trace(r, any_hit=any_hit)
            if any_hit:
                assert np.array_equal(h["id"] >= 0, ref["id"] >= 0), shape
            else:
                assert np.array_equal(h["id"], ref["id"]), shape
    s.free()
