"""What a server makes of its device memory budget: two-part passes under every traversal configuration, and no part of
the budget set aside for nothing."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu


def kernels(fn):
    """Kernel launches of fn() by name."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return {e.key: e.count for e in p.key_averages()}


# the default, shapes with more resident threads than it, a refilled one and the reference layout
@pytest.mark.parametrize("cfg", [(256, 16, 64, 0, 0), (64, 8, 64, 0, 0), (64, 8, 64, 0, 1), (256, 16, 64, 1, 0)])
def test_a_configured_server_keeps_its_two_parts(cfg):
    s = gpr.Scene.sphere_grid(8, 8, 4)
    c = gpr.lookat((0, 0, 0), (1.0, 6, 9))
    srv = gpr.Server(gpr.arena_bytes(s) + (4 << 30), gpr.arena_bytes(s), capacity=1 << 21, max_jobs=4)
    job = gpr.job(srv.add_scene(s), 512, 512, 8, c, 40, 3, 3, 7)
    print(f"[server] parts {cfg}", flush=True)
    want = srv.wait(srv.submit(job))[0]
    srv.set_cfg(*cfg)
    got = [srv.wait(srv.submit(job))[0]]  # captures the pass
    n = kernels(lambda: got.append(srv.wait(srv.submit(job))[0]))
    gen = sum(v for k, v in n.items() if "k_gen" in k)
    assert gen == 2, n
    if cfg[3] == 0:
        for g in got:
            assert np.array_equal(g.view(np.uint32), want.view(np.uint32))
    srv.free()
