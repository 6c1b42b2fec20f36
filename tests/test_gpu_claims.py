"""Turns claimed from several counters: every ray of a batch is traced, whatever the number of waves and turns."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

QUAD_RAYS = 1 << 17  # default launch shape: four lanes to a ray up to here


@pytest.mark.parametrize("n", [1, 7, 64 * 7 + 1, 200001, 1000003])
@pytest.mark.parametrize("cfg", [None, (64, 8, 64, 0), (512, 32, 512, 0), (64, 16, 64, 1), (512, 8, 4096, 1)])
def test_every_ray_is_traced(n, cfg):
    import torch
    print(f"[claims] {n} rays cfg {cfg}", flush=True)
    s = gpr.Scene.soup(gpr.gen_soup(5, 0, 500, 0.05)).commit()
    r = torch.zeros(n, 8, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(n)
    r[:, 0:3] = torch.rand(n, 3, generator=g, device="cuda")
    r[:, 3:6] = torch.randn(n, 3, generator=g, device="cuda")
    r[:, 7] = float("inf")
    hits = torch.full((n, 4), float("nan"), device="cuda")
    if cfg:
        s.trace_set_cfg(*cfg)
    s.trace_device(r.data_ptr(), hits.data_ptr(), n)
    torch.cuda.synchronize()
    assert not torch.isnan(hits[:, 0]).any()
    # the same rays in calls of the short-batch form
    want = torch.empty_like(hits)
    t = gpr.Scene.soup(gpr.gen_soup(5, 0, 500, 0.05)).commit()
    for a in range(0, n, QUAD_RAYS):
        m = min(QUAD_RAYS, n - a)
        t.trace_device(r[a:].data_ptr(), want[a:].data_ptr(), m)
    torch.cuda.synchronize()
    assert torch.equal(hits.view(torch.int32), want.view(torch.int32))
    s.free()
    t.free()
