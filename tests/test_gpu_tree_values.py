"""The build's own checks (every parent box is the union of its children's, bit for bit) accept what the build makes of
unusual coordinates: zeros of both signs, subnormal and huge numbers, infinities, NaN; the tree is the oracle's."""
import numpy as np
import pytest

import gpr
import oracle_py as O

pytestmark = pytest.mark.gpu


def positions(kind, n):
    g = np.random.default_rng(n)
    p = g.random((n, 9), dtype=np.float32) - np.float32(0.5)
    if kind == "zeros":
        p[:] = np.where(g.random(p.shape) < 0.5, np.float32(0), np.float32(-0.0))
        p[::3] += g.random((len(p[::3]), 9), dtype=np.float32)
    elif kind == "subnormal":
        p *= np.float32(1e-41)
    elif kind == "huge":
        p *= np.float32(3e38)
    elif kind == "infinite":
        p[n // 3, 4], p[n // 2, 2] = np.inf, -np.inf
    else:
        p[::7, 4] = np.nan
    return p


@pytest.mark.parametrize("kind", ["zeros", "subnormal", "huge", "infinite", "nan"])
@pytest.mark.parametrize("n", [2, 511, 512, 513, 5000, 70001])
def test_unusual_coordinates(kind, n):
    p = positions(kind, n)
    print(f"[tree] {kind} {n}", flush=True)
    s = gpr.Scene.soup(p).commit()
    assert np.array_equal(s.ref_layout().view(np.uint32), O.lbvh(p)[0].view(np.uint32))
    s.free()
