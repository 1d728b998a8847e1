"""Rader over two passes: a prime of every column length that has the compiled gather
and scatter (128, 256, 512, 1000, 1008, 1024) and of one that has none, out of place
(x[0] read and X[0] stored by the passes), in place and real, against numpy's float64
transforms.  Bars as in the other GPU tests: 1e-12 log2 N (double), 5e-7 log2 N (float).
"""
import math

import numpy as np
import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, dtype=np.complex128), np.asarray(b, dtype=np.complex128)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("p,cols", [(17921, 128), (76801, 256), (262657, 512), (1008001, 1000),
                                    (1032193, 1008), (1053697, 1024), (12289, 96)])
def test_two_pass_rader(p, cols, half):
    import torch

    rng = np.random.default_rng(p)
    b = 3 if p < 100000 else 2
    bar = (5e-7 if half else 1e-12) * math.log2(p)
    x = (rng.uniform(-1, 1, (b, p)) + 1j * rng.uniform(-1, 1, (b, p)) + 2.0)
    x = x.astype(np.complex64 if half else np.complex128)
    xd = torch.from_numpy(x).cuda()
    for flags, f in ((0, np.fft.fft), (K.FLAG_INVERSE, np.fft.ifft)):
        plan = K.CpxPlan(p, flags, half=half)
        assert f"four-step {cols}x" in plan.describe()
        ref = f(x.astype(np.complex128))
        got = plan(xd)
        assert rel(got.cpu().numpy(), ref) <= bar
        assert rel(got[:, 0].cpu().numpy(), ref[:, 0]) <= bar
        inplace = xd.clone()
        plan(inplace, inplace)
        assert rel(inplace.cpu().numpy(), ref) <= bar
        assert rel(inplace[:, 0].cpu().numpy(), ref[:, 0]) <= bar
    r = np.ascontiguousarray(x.real)
    X = K.ScalarPlan(p, half=half).forward(r)
    assert rel(X, np.fft.fft(r.astype(np.float64))) <= bar
    back = K.ScalarPlan(p, K.FLAG_INVERSE, half=half).inverse(X)
    assert rel(back, r) <= 2 * bar
    assert rel(back[:, 0], r[:, 0]) <= 4 * bar
