"""Skewed keys: buckets too large for LDS are sorted in pieces by several blocks.  Against a stable sort on the host, at
sizes where a bucket turns large, with sub-buckets above and below what is placed by rank, through both entry points."""
import numpy as np
import pytest

import gpr

pytestmark = pytest.mark.gpu


def keys_of(kind, n, g):
    k = g.integers(0, 1 << 30, n)
    if kind == "clusters":        # dense objects in a large scene: 64 values of the upper bits in use, all of them small
        k = (k & 0x7FFF) | ((k >> 24) << 15)
    elif kind == "outlier":       # one cluster and a far point
        k = k & 0x3FFFF
        k[n // 3] = (1 << 30) - 1
    elif kind == "equal":
        k[:] = 0x2ABCDEF1
    elif kind == "two":
        k = np.where(k & 1, 5, (1 << 29) + 7)
    elif kind == "crowded":       # sub-buckets of thousands of keys that differ below
        k = (k & 0x3FF) | (((k >> 12) & 0x3) << 20) | (((k >> 20) & 1) << 29)
    elif kind == "mixed":         # a uniform half, a cluster, and equal keys
        k[n // 2:] &= 0xFFFF
        k[-n // 8:] = 77
    return k.astype(np.uint32)


@pytest.mark.parametrize("kind", ["clusters", "outlier", "equal", "two", "crowded", "mixed"])
@pytest.mark.parametrize("n", [1536, 1537, 3100, 8191, 40003, 399952, 1 << 20])
def test_skewed_keys(kind, n):
    import torch
    g = np.random.default_rng(n)
    k = keys_of(kind, n, g)
    order = np.argsort(k, kind="stable")
    dk = torch.from_numpy(k.view(np.int32)).cuda()
    uni = torch.from_numpy(g.integers(0, 1 << 30, n).astype(np.int32)).cuda()
    for fn in (gpr.sort_pairs_device, gpr.sort_pairs_device_noalloc):
        print(f"[skew] {kind} {n} {fn.__name__}", flush=True)
        for keys in (dk, uni, dk):  # a call leaves the next one's counters cleared
            sk, si = torch.empty_like(keys), torch.empty_like(keys)
            fn(keys.data_ptr(), sk.data_ptr(), si.data_ptr(), n)
        torch.cuda.synchronize()
        assert np.array_equal(sk.cpu().numpy().view(np.uint32), k[order])
        assert np.array_equal(si.cpu().numpy(), order.astype(np.int32))
