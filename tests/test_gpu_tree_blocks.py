"""The LBVH build around the runs of leaves that one block builds on the GPU: sizes next to multiples of 512 and 4096
leaves, runs of equal keys that cross a block's edge, trees deeper than a block."""
import numpy as np
import pytest

import gpr
import gpu_scenes as G
import oracle_py as O

pytestmark = pytest.mark.gpu


def runs(n, seed=7):
    """Equal-key runs of 1 to 1,400 leaves, in key order along a diagonal."""
    rng = np.random.default_rng(seed)
    c, k = [], 0
    while k < n:
        m = int(rng.choice([1, 2, 3, 40, 600, 1400]))
        c += [rng.random()] * m
        k += m
    c = np.asarray(c[:n], np.float32)[:, None, None]
    d = np.array([[0, 0, 0], [1e-5, 0, 0], [0, 1e-5, 0]], np.float32)
    return (c + d + np.arange(n, dtype=np.float32)[:, None, None] * np.float32(1e-9)).reshape(n, 9).astype(np.float32)


KINDS = {"soup": G.soup, "duplicates": G.duplicate_heavy, "identical": G.identical, "collinear": G.collinear, "runs": runs}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("n", [1, 2, 3, 5, 511, 512, 513, 1023, 1025, 4095, 4097, 9000])
def test_tree_at_block_edges(kind, n):
    pos = KINDS[kind](n)
    print(f"[tree] {kind} {n}", flush=True)
    s = G.scene_from_soup(pos)
    nodes, sk, si = O.lbvh(pos)
    _, gsk, gsi = s.keys()
    assert np.array_equal(gsk, sk) and np.array_equal(gsi, si)
    assert np.array_equal(s.ref_layout().view(np.uint32), nodes.view(np.uint32))
    # the four-wide tree holds every triangle: it hits what the reference layout hits
    r = gpr.gen_rays(6, 1, 600)
    c = pos.reshape(-1, 3, 3).mean(1)
    r["o"] = np.random.default_rng(1).random((600, 3))
    r["d"] = c[np.random.default_rng(2).integers(0, n, 600)] - r["o"]
    fast, ref = s.trace(r), s.trace(r, ref_order=True)
    assert np.array_equal(fast["id"] >= 0, ref["id"] >= 0)
    first = s.info().bvh4_nodes
    s.build()  # again into the same memory
    assert s.info().bvh4_nodes == first
    assert np.array_equal(s.ref_layout().view(np.uint32), nodes.view(np.uint32))
    s.free()
