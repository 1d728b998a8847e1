"""Real 2D convolution on both sides of the column count from which the longest
columns run in one pass (64 and 65 columns), and with one column pair, against numpy's
float64 transforms.  Bars as in the other GPU tests: 1e-12 log2 N (double), 5e-7 log2 N
(float)."""
import math

import numpy as np
import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("y", [4000, 4160])
@pytest.mark.parametrize("x", [2, 126, 128])
def test_columns_near_the_width(x, y, half):
    rng = np.random.default_rng(x * 10000 + y)
    t = np.float32 if half else np.float64
    a, b = (rng.uniform(-1, 1, (y, x)).astype(t) for _ in range(2))
    ref = np.fft.irfft2(np.fft.rfft2(a.astype(np.float64)) * np.fft.rfft2(b.astype(np.float64)),
                        s=(y, x))
    got = K.Conv2Plan(x, y, real=True, half=half)(a, b)
    bar = (5e-7 if half else 1e-12) * math.log2(x * y)
    assert np.linalg.norm(got - 2 * ref) <= 2 * bar * np.linalg.norm(2 * ref)
