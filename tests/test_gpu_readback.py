"""Read-back of the radiance sums: packed on the device in chunks of 2^20 pixels.
The pixels are planted with restore(), so the copy has to return the same bits."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (17, 3), (1024, 1024), (1025, 1024), (1531, 1401)])
def test_read_returns_the_bits_of_the_frame_buffer(w, h):
    print(f"[readback] {w}x{h}", flush=True)
    r = gpr.Renderer(gpr.Scene.cornell(w, h), max_depth=2, rng_mode=gpr.RNG_PCG)
    rgb = np.random.default_rng(w).integers(0, 1 << 32, (w * h, 3), dtype=np.uint32).view(np.float32)
    r.restore(rgb, 3)
    for _ in range(2):
        got, cnt = r.read()
        assert np.array_equal(got.view(np.uint32), rgb.view(np.uint32))
        assert (cnt == 3).all()

