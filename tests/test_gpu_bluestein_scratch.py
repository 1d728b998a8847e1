"""Scratch of Bluestein lengths: a batch needs no more of it, in the fixed array of
the allocation-free entry point and under a device-memory budget, than the shortest
2,3,5-smooth convolution length takes, whichever convolution length the plan runs.
"""
import os
import re

import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu

LIMIT = 32 << 20


def shortest(n):
    m = 2 * n - 1
    while True:
        r = m
        for p in (2, 3, 5):
            while r % p == 0:
                r //= p
        if r == 1:
            return m
        m += 1


def data(b, n, half):
    import torch

    g = torch.Generator(device="cuda").manual_seed(n)
    t = torch.float32 if half else torch.float64
    return torch.view_as_complex(torch.rand(b, n, 2, generator=g, device="cuda", dtype=t) - 0.5)


@pytest.mark.parametrize("n,half", [(94132, False), (33331, False), (33331, True), (1069, False),
                                    (300017, False)])
def test_noalloc_takes_the_batches_of_the_shortest_length(n, half):
    import torch

    each = shortest(n) * (8 if half else 16)
    most = (LIMIT - 256) // each
    p = K.CpxPlan(n, half=half)
    x = data(most + 1, n, half)
    ref = torch.empty_like(x)
    torch.cuda.synchronize()
    p.run_async(x, ref, most)
    K.synchronize(half)
    got = torch.zeros_like(x)
    torch.cuda.synchronize()
    p.run_noalloc(x, got, most)
    K.synchronize(half)
    assert torch.equal(got[:most], ref[:most])
    # rows shifted by one in one buffer, in groups of the batch where they do not fit at once
    for src, dst in ((0, 1), (1, 0)):
        buf = x.clone()
        rows = buf[src:src + most].clone()
        torch.cuda.synchronize()  # (the library's stream does not wait for torch's)
        p.run_async(rows, ref, most)
        p.run_noalloc(buf[src:], buf[dst:], most)
        K.synchronize(half)
        assert torch.equal(buf[dst:dst + most], ref[:most])
    with pytest.raises(K.KfftError, match="limit"):
        p.run_noalloc(x, got, most + 1)


def _held(p, x, y, b):
    """Bytes the library holds, from the text of a refused call (nothing launched)."""
    os.environ["KFFT_AMD_DEVICE_LIMIT_MB"] = "1"
    assert p.L.kfft_eval_cpx_batch_async(p.handle, K._ptr(x), K._ptr(y), b, None) == K.RET_GPU_FAIL
    return int(re.search(r"(\d+) held", K.last_error(p.half)).group(1))


@pytest.mark.parametrize("n,half,b", [(33331, False, 64), (94132, True, 50)])
def test_batch_within_a_budget_for_the_shortest_length(n, half, b):
    import torch

    p, q = K.CpxPlan(n, half=half), K.CpxPlan(n, half=half)
    x = data(b, n, half)
    ref, y = torch.empty_like(x), torch.empty_like(x)
    torch.cuda.synchronize()
    p.run_async(x, ref, b)
    K.synchronize(half)
    try:
        held = _held(q, x, y, b)
        need = b * shortest(n) * (8 if half else 16)
        os.environ["KFFT_AMD_DEVICE_LIMIT_MB"] = str(((held + need) >> 20) + 1)
        q.run_async(x, y, b)
    finally:
        del os.environ["KFFT_AMD_DEVICE_LIMIT_MB"]
    K.synchronize(half)
    assert torch.equal(y, ref)


def test_plan_within_a_budget_for_the_shortest_length():
    """A budget that the shortest length's tables (19 MiB at most while they are made)
    and scratch fit into, but not the power of two's (44 MiB)."""
    import torch

    n = 133526  # (a length no other test plans): 270000 points, or 2^19
    x, w = data(1, n, False), data(8, 65536, False)
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    try:
        held = _held(K.CpxPlan(65536), w, w, 8)
        os.environ["KFFT_AMD_DEVICE_LIMIT_MB"] = str((held >> 20) + 30)
        p = K.CpxPlan(n)
        p.run_async(x, y, 1)
    finally:
        del os.environ["KFFT_AMD_DEVICE_LIMIT_MB"]
    K.synchronize(False)
    assert f"inner={shortest(n)} " in p.describe()
    ref = K.CpxPlan(n)(x)
    assert float((y - ref).norm() / ref.norm()) < 2e-14
