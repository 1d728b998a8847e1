"""Real transforms whose output lies over their own input (one device buffer for
both, rows of n reals against rows of n/2+1 or n bins), and complex rows shifted by
one row in one buffer: every row is read before anything is stored over it, at any
batch.  One-pass, long one-pass (a row per CU), two-pass, Rader and Bluestein
lengths, against numpy's float64 transforms.

Bars as in the other GPU tests: 1e-12 log2 N (double), 5e-7 log2 N (float).
"""
import math
import os
import re

import numpy as np
import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, dtype=np.complex128), np.asarray(b, dtype=np.complex128)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def bar(n, half):
    return (5e-7 if half else 1e-12) * max(1.0, math.log2(n))


# half lengths with the long one-pass rows, then one-pass (compiled and not), two-pass;
# odd: one pass, Bluestein, Rader
CASES = ([(2 * h, False, 300) for h in (5120, 6144, 6250, 6400, 6561, 7680, 8192)]
         + [(2 * h, True, 300) for h in (10000, 10240, 15360)]
         + [(n, half, 41) for n in (128, 512, 2000, 2310, 4096, 16384, 65536) for half in (False, True)]
         + [(n, half, 41) for n in (105, 111, 1009, 4355) for half in (False, True)])


@pytest.mark.parametrize("n,half,batch", CASES)
def test_forward_real_over_its_input(n, half, batch):
    import torch

    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (batch, n)).astype(np.float32 if half else np.float64)
    ctype = torch.complex64 if half else torch.complex128
    full = np.fft.fft(x.astype(np.float64))
    for flags in (0, K.FLAG_EXPAND_SCALAR):
        p = K.ScalarPlan(n, flags, half=half)
        buf = torch.zeros(batch * p.out_len, dtype=ctype, device="cuda")
        torch.view_as_real(buf).reshape(-1)[:batch * n] = torch.from_numpy(x).cuda().reshape(-1)
        torch.cuda.synchronize()
        assert p.L.kfft_eval_scalar_batch(p.handle, buf.data_ptr(), buf.data_ptr(), batch) == 0
        got = buf.view(batch, p.out_len).cpu().numpy()
        assert rel(got, full[:, :p.out_len]) <= bar(n, half), flags


@pytest.mark.parametrize("n,half,batch", [c for c in CASES if c[0] % 2])
def test_inverse_real_over_its_input(n, half, batch):
    import torch

    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (batch, n)).astype(np.float32 if half else np.float64)
    X = np.fft.fft(x.astype(np.float64)).astype(np.complex64 if half else np.complex128)
    p = K.ScalarPlan(n, K.FLAG_INVERSE, half=half)
    buf = torch.from_numpy(X).cuda()
    assert p.L.kfft_evali_scalar_batch(p.handle, buf.data_ptr(), buf.data_ptr(), batch) == 0
    got = torch.view_as_real(buf).reshape(-1)[:batch * n].view(batch, n).cpu().numpy()
    assert rel(got, x) <= 2 * bar(n, half)


def test_forward_real_over_its_input_within_a_budget():
    """No room for the rows in scratch: the passes run as on separate buffers (two-pass
    lengths are right there too up to one group of transforms)."""
    import torch

    n, batch = 2 * 6561, 300
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (batch, n))
    p = K.ScalarPlan(n)
    buf = torch.zeros(batch * p.out_len, dtype=torch.complex128, device="cuda")
    torch.view_as_real(buf).reshape(-1)[:batch * n] = torch.from_numpy(x).cuda().reshape(-1)
    torch.cuda.synchronize()
    run = lambda: p.L.kfft_eval_scalar_batch(p.handle, buf.data_ptr(), buf.data_ptr(), batch)  # noqa: E731
    try:
        os.environ["KFFT_AMD_DEVICE_LIMIT_MB"] = "1"
        assert run() == K.RET_GPU_FAIL  # (nothing launched: the text says what is held)
        held = int(re.search(r"(\d+) held", K.last_error(False)).group(1))
        # the passes' scratch takes 30 MiB, with the rows in scratch 60
        os.environ["KFFT_AMD_DEVICE_LIMIT_MB"] = str((held >> 20) + 40)
        assert run() == 0
    finally:
        del os.environ["KFFT_AMD_DEVICE_LIMIT_MB"]
    assert rel(buf.view(batch, p.out_len).cpu().numpy(), np.fft.rfft(x)) <= bar(n, False)


def test_complex_rows_shifted_by_one():
    import torch

    n, batch = 6561, 300
    g = torch.Generator(device="cuda").manual_seed(1)
    buf = torch.view_as_complex(torch.rand((batch + 1) * n, 2, generator=g, device="cuda",
                                           dtype=torch.float64) - 0.5)
    p = K.CpxPlan(n)
    for src, dst in ((0, n), (n, 0)):
        x = buf[src:src + batch * n].view(batch, n).cpu().numpy()
        torch.cuda.synchronize()
        p(buf[src:src + batch * n].view(batch, n), buf[dst:dst + batch * n].view(batch, n))
        got = buf[dst:dst + batch * n].view(batch, n).cpu().numpy()
        assert rel(got, np.fft.fft(x)) <= bar(n, False)
