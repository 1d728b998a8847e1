"""Blocking calls are ordered after work on the caller's blocking streams: a buffer that
a stream made with hipStreamCreate still fills, with nothing on the null stream itself,
is complete when a blocking call reads it."""
import ctypes

import numpy as np
import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1024, 94132])
def test_blocking_call_waits_for_a_blocking_stream(n):
    import torch

    hip = ctypes.CDLL("libamdhip64.so")
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    side = torch.cuda.ExternalStream(handle.value)
    p = K.CpxPlan(n)
    big = torch.rand(4096, 4096, device="cuda")
    prod = torch.empty_like(big)
    x = torch.zeros(n, 2, device="cuda", dtype=torch.float64)
    out = torch.empty(n, device="cuda", dtype=torch.complex128)
    src = torch.linspace(-1, 1, 2 * n, device="cuda", dtype=torch.float64).view(n, 2)
    p(torch.view_as_complex(x), out)
    torch.cuda.synchronize()
    ref = np.fft.fft(torch.view_as_complex(src).cpu().numpy())
    for _ in range(3):
        x.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(30):
                torch.mm(big, big, out=prod)
            x.copy_(src)
        p(torch.view_as_complex(x), out)
        got = out.cpu().numpy()
        assert np.linalg.norm(got - ref) <= 1e-12 * np.log2(n) * np.linalg.norm(ref)
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0
