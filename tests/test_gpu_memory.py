"""Device memory.  Passes of several samples on a device that has little left: they get smaller, the images keep their
bits, nothing is allocated over and over, and nothing is held that is of no use.  What a server makes of its budget: two-part
passes under every traversal configuration, none of it set aside for nothing, and small budgets accepted."""
import contextlib

import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

GB = 1 << 30


@contextlib.contextmanager
def left(nbytes):
    """All device memory but nbytes is taken."""
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    t = []
    try:
        for _ in range(4):  # one large allocation can leave more than it should
            more = torch.cuda.mem_get_info()[0] - nbytes
            if more < 32 << 20:
                break
            t.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        print(f"[memory] {torch.cuda.mem_get_info()[0] >> 20} MiB left", flush=True)
        yield
    finally:
        torch.cuda.synchronize()
        t.clear()
        torch.cuda.empty_cache()


def calls(fn):
    """Runtime calls and kernel launches of fn() by name."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return {e.key: e.count for e in p.key_averages()}


def bits(a):
    return a.view(np.uint32)


def renderer(scene):
    r = gpr.Renderer(scene, max_depth=8, rr_start=3, seed=5)
    r.render(1)  # what a render of one sample holds
    r.reset()
    return r


# 4 samples of 1920x1080 at depth 8 take buffers of 4.2 GB, 2 take 2.1
def test_smaller_passes_are_kept():
    s = gpr.Scene.sphere_grid(1920, 1080, 4)
    one = renderer(s)
    for _ in range(4):
        one.render(1)
    want = one.read()[0]
    one.free()
    r = renderer(s)
    with left(3 * GB):
        r.render(4)
        assert np.array_equal(bits(r.read()[0]), bits(want))

        def again():
            r.reset()
            r.render(4)

        n = calls(again)
        accum = sum(v for k, v in n.items() if "k_accum" in k)
        assert accum == 2, n  # two passes of two samples
        busy = [k for k in n if "hipMalloc" in k or "hipFree" in k or "GraphInstantiate" in k]
        assert not busy, n
        assert np.array_equal(bits(r.read()[0]), bits(want))
    again()  # and with room for all four again
    assert sum(v for k, v in calls(again).items() if "k_accum" in k) == 1
    assert np.array_equal(bits(r.read()[0]), bits(want))
    r.free()


def test_no_room_holds_nothing():
    import torch
    s = gpr.Scene.sphere_grid(1920, 1080, 4)
    r = renderer(s)
    with left(GB + GB * 3 // 10):
        before = torch.cuda.mem_get_info()[0]
        r.render(2)
        assert abs(torch.cuda.mem_get_info()[0] - before) < 64 << 20
    r.free()


# 4 samples of 1024x1024 at depth 8 take term lists of 1.14 GB, 2 take 0.57
def test_a_batch_keeps_smaller_passes():
    s = gpr.Scene.sphere_grid(8, 8, 4)

    def batch():
        b = gpr.Batch(gpr.arena_bytes(s), capacity=1 << 22, max_jobs=4)
        b.add_job(gpr.job(b.add_scene(s), 1024, 1024, 16, gpr.lookat((0, 0, 0), (1.0, 6, 9)), 40, 8, 3, 7))
        return b

    b = batch()
    b.run()
    want = b.read(0)
    b.free()
    b = batch()
    with left(GB * 9 // 10):
        b.run()
        assert np.array_equal(bits(b.read(0)), bits(want))
        n = calls(b.run)
        assert sum(v for k, v in n.items() if "k_accum" in k) == 8, n
        assert np.array_equal(bits(b.read(0)), bits(want))
    b.free()


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
    n = calls(lambda: got.append(srv.wait(srv.submit(job))[0]))
    gen = sum(v for k, v in n.items() if "k_gen" in k)
    assert gen == 2, n
    if cfg[3] == 0:
        for g in got:
            assert np.array_equal(g.view(np.uint32), want.view(np.uint32))
    srv.free()


# budgets from the smallest accepted one up: none, a few and many bytes a path beyond the queues and four passes of frames
@pytest.mark.parametrize("bytes_a_path", [17, 40, 70, 100, 127, 140, 300])
def test_a_server_uses_its_whole_budget(bytes_a_path):
    import torch
    arena, capacity = 1 << 20, 1 << 22

    def used(budget):
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        srv = gpr.Server(budget, arena, capacity=capacity, max_jobs=4)
        after = torch.cuda.mem_get_info()[0]
        srv.free()
        return before - after

    lo, hi = 0, 4 << 30  # the smallest accepted budget: arena, queues and a frame of the capacity
    while hi - lo > 1 << 16:
        mid = (lo + hi) // 2
        try:
            gpr.Server(mid, arena, capacity=capacity, max_jobs=4).free()
            hi = mid
        except gpr.GprError:
            lo = mid
    budget = hi - 16 * capacity + bytes_a_path * capacity
    got = used(budget)
    print(f"[server] {bytes_a_path} B a path: budget {budget >> 20} MiB, in use {got >> 20}", flush=True)
    # allocations are whole 2-MiB pages, some twenty of them; streams and events take a few more
    assert budget - (48 << 20) < got < budget + (64 << 20)


# the smallest budgets that servers of these capacities were accepted with before passes had two parts and eight claim
# counters, with 1 MiB of arena and 256 compute units
@pytest.mark.parametrize("capacity,budget", [(1000, 2289165), (10000, 11689485), (65536, 68484621), (131072, 135724557),
                                             (262144, 270204429), (500000, 482566669), (655360, 522649101),
                                             (1048576, 624098829), (1310720, 691731981), (4194304, 1435696653)])
def test_small_budgets_are_accepted(capacity, budget):
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the stack overflow area depends on the number of compute units")
    gpr.Server(budget, 1 << 20, capacity=capacity, max_jobs=4).free()
