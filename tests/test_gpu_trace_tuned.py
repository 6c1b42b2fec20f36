"""A tuned scene: short batches walk a ray with four lanes as on a scene that was not tuned, whatever the tuner was given;
a configuration that the caller sets holds for all of them; hits are the same."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu

QUAD = 1 << 17


def kernels(fn):
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return " ".join(e.key for e in p.key_averages())


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("tuned_on", [2000, QUAD, QUAD + 1, 1 << 20])
def test_short_batches_of_a_tuned_scene(tuned_on, any_hit):
    import torch
    s = gpr.Scene.soup(gpr.gen_soup(3, 0, 20000, 0.02)).commit()
    rays = gpr.gen_rays(3, 1, max(tuned_on, QUAD + 1))
    if any_hit:
        rays = gpr.gen_shadow_rays(3, 2, rays)
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()

    def hits(n):
        out = torch.zeros(n, 4, device="cuda")
        s.trace_device(d.data_ptr(), out.data_ptr(), n, any_hit=any_hit)
        torch.cuda.synchronize()
        return out.cpu().numpy().view(np.uint32)

    sizes = (1, 2000, QUAD, QUAD + 1)
    want = [hits(n) for n in sizes]
    print(f"[tuned] on {tuned_on} any {any_hit}", flush=True)
    best = s.trace_tune(d.data_ptr(), tuned_on, any_hit=any_hit)[0]
    for n, w in zip(sizes, want):
        assert np.array_equal(hits(n), w), n
        assert ("k_trace_quad" in kernels(lambda: hits(n))) == (n <= QUAD), n
    s.trace_set_cfg(best.block, best.stack, best.chunk, best.refill)
    for n, w in zip(sizes, want):
        assert np.array_equal(hits(n), w), n
        assert "k_trace_quad" not in kernels(lambda: hits(n)), n
