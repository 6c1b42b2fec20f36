"""Ordered queues of reference RNG mode: tiles of 512 entries, 64 of them to a look-back step.  The image and the queue
sizes have to be the serial order's, at sizes around a tile, a step and a partial last tile."""
import numpy as np
import pytest

import gpr
from test_gpu_render import gpu_render, oracle_render

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (511, 1), (512, 1), (513, 1), (256, 128), (257, 128), (331, 199)])
def test_ordered_appends(w, h):
    s = gpr.Scene.sphere_grid(w, h, 3)
    print(f"[ordered] {w}x{h}", flush=True)
    got, cnt, _, _ = gpu_render(s, 2, 3, gpr.RNG_REFERENCE, 3, gpr.TRAVERSAL_REF)
    want, wcnt = oracle_render(s, 2, 3, gpr.RNG_REFERENCE, 3)
    assert np.array_equal(cnt, wcnt)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
