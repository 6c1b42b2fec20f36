"""Sorts of many keys: from 3 * 2^20 on with larger pieces of a bucket, from 15 * 2^20 on by three stable passes.  The
result is checked against its definition (keys ascending, ties by index, every index once), on the device; and a sort of
skewed keys may not cost a multiple of one of uniform keys where the stable passes take over."""
import pytest

import gpr

pytestmark = pytest.mark.gpu

WIDE, RADIX = 3 << 20, 15 << 20


def keys_of(kind, n):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    k = torch.randint(0, 1 << 30, (n,), generator=g, device="cuda", dtype=torch.int32)
    if kind == "clusters":   # dense objects in a large scene
        k = (k & 0x7FFF) | ((k >> 24) << 15)
    elif kind == "equal":
        k[:] = 0x2ABCDEF1
    elif kind == "crowded":  # sub-buckets of thousands of keys that differ below, and the largest key
        k = (k & 0x3FF) | (((k >> 12) & 0x3) << 20) | (((k >> 20) & 1) << 29)
        k[n // 3] = (1 << 30) - 1
    return k


def run(k, sk, si):
    gpr.sort_pairs_device(k.data_ptr(), sk.data_ptr(), si.data_ptr(), k.numel())


def check(k, sk, si):
    import torch
    n = k.numel()
    assert bool((k[si.long()] == sk).all())
    assert bool(((sk[1:] > sk[:-1]) | ((sk[1:] == sk[:-1]) & (si[1:] > si[:-1]))).all())
    seen = torch.zeros(n, dtype=torch.int32, device="cuda").index_add_(0, si, torch.ones_like(si))
    assert bool((seen == 1).all())


@pytest.mark.parametrize("kind", ["uniform", "clusters", "equal", "crowded"])
@pytest.mark.parametrize("n", [WIDE, WIDE + 1, 4000003, RADIX, RADIX + 1, RADIX + 8192 * 5, 20000003])
def test_many_keys(kind, n):
    import torch
    if kind in ("equal", "crowded") and WIDE + 1 < n <= RADIX:
        n = 4000003  # pieces of one bucket: quadratic in its keys, so the small end
    print(f"[sort] {kind} {n}", flush=True)
    k = keys_of(kind, n)
    sk, si = torch.full_like(k, -1), torch.full_like(k, -1)
    run(k, sk, si)
    check(k, sk, si)
    # a call leaves the next one's counters cleared, whichever path each takes
    u = keys_of("uniform", 100003)
    usk, usi = torch.full_like(u, -1), torch.full_like(u, -1)
    run(u, usk, usi)
    check(u, usk, usi)


def test_many_keys_captured():
    import torch
    st = torch.cuda.Stream()
    k = keys_of("clusters", RADIX + 4097)
    sk, si = torch.empty_like(k), torch.empty_like(k)
    print("[sort] captured", flush=True)
    with torch.cuda.stream(st):
        gpr.set_stream(st.cuda_stream)
        try:
            run(k, sk, si)  # allocates the stream's scratch
            st.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=st):
                run(k, sk, si)
            for r in range(3):
                k.copy_(keys_of("uniform", k.numel()) ^ r)
                sk.fill_(-1)
                si.fill_(-1)
                graph.replay()
                st.synchronize()
                check(k, sk, si)
        finally:
            gpr.set_stream(0)
            gpr.release_stream(st.cuda_stream)


@pytest.mark.parametrize("n", [RADIX + 1, 1 << 24])
def test_cost_of_skewed_keys(n):
    import torch
    ms = {}
    for kind in ("uniform", "clusters", "equal"):
        print(f"[sort] cost {kind} {n}", flush=True)
        k = keys_of(kind, n)
        sk, si = torch.empty_like(k), torch.empty_like(k)
        run(k, sk, si)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        run(k, sk, si)
        b.record()
        b.synchronize()
        ms[kind] = a.elapsed_time(b)
    print(ms, flush=True)
    assert ms["clusters"] < 4 * ms["uniform"] and ms["equal"] < 4 * ms["uniform"], ms
