"""The shaped general passes compiled per use: Bluestein's (one pass, and the
three passes of a two-pass convolution length) at the smallest and largest
length of every power-of-two convolution length, Rader's one-pass form, both
directions, real and complex data, partial tiles and in place, against numpy's
float64 transforms; and the order of blocking calls with earlier work.

Bars as in the other GPU tests: 1e-12 log2 N (double), 5e-7 log2 N (float).
"""
import math

import numpy as np
import pytest

import kfft_amd as K

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, dtype=np.complex128), np.asarray(b, dtype=np.complex128)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def bar(n, half):
    return (5e-7 if half else 1e-12) * max(1.0, math.log2(n))


def smooth31(n):
    for p in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31):
        while n % p == 0:
            n //= p
    return n == 1


def is_prime(n):
    return n > 1 and all(n % d for d in range(2, int(n ** 0.5) + 1))


def chirped(n):  # a length that runs Bluestein
    return not smooth31(n) and not (is_prime(n) and smooth31(n - 1))


def edges(lg):
    """First and last Bluestein length whose power-of-two convolution length is 2^lg."""
    lo, hi = (1 << (lg - 2)) + 1, 1 << (lg - 1)
    return (next(n for n in range(lo, hi + 1) if chirped(n)),
            next(n for n in range(hi, lo - 1, -1) if chirped(n)))


def batch_of(n):
    return 1 if n > 60000 else 3 if n > 3000 else 37


def data(rng, half, *shape):
    x = rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)
    return x.astype(np.complex64) if half else x


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lg", range(8, 21))
def test_bluestein_lengths(lg, half):
    for n in edges(lg):
        rng = np.random.default_rng(n)
        x = data(rng, half, batch_of(n), n)
        x64 = x.astype(np.complex128)
        assert rel(K.CpxPlan(n, half=half)(x), np.fft.fft(x64)) <= bar(n, half), n
        y = K.CpxPlan(n, K.FLAG_INVERSE, half=half)(x)
        assert rel(y, np.fft.ifft(x64)) <= bar(n, half), n


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lg", [8, 11, 12, 13, 14, 16])
def test_bluestein_real(lg, half):
    """Odd lengths (real rows through the chirped pass) and twice an edge length
    (the half-length transform with the separate rebuild)."""
    lo, hi = edges(lg)
    odd = next(n for n in range(lo, hi) if n % 2 and chirped(n))
    for n in (odd, 2 * hi):
        rng = np.random.default_rng(n)
        x = rng.uniform(-1, 1, (batch_of(n), n)).astype(np.float32 if half else np.float64)
        ref = (np.fft.fft if n % 2 else np.fft.rfft)(x.astype(np.float64))
        X = K.ScalarPlan(n, half=half).forward(x)
        assert rel(X, ref) <= bar(n, half), n
        back = K.ScalarPlan(n, K.FLAG_INVERSE, half=half).inverse(X)
        assert rel(back, x.astype(np.float64) * (1 if n % 2 else 2)) <= 2 * bar(n, half), n


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n", [257, 1009, 2081])
@pytest.mark.parametrize("batch", [1, 2, 5])
def test_rader_one_pass(n, batch, half):
    import torch

    rng = np.random.default_rng(n + batch)
    x = data(rng, half, batch, n)
    xd = torch.from_numpy(x).cuda()
    for flags, f in ((0, np.fft.fft), (K.FLAG_INVERSE, np.fft.ifft)):
        p = K.CpxPlan(n, flags, half=half)
        ref = f(x.astype(np.complex128))
        assert rel(p(xd).cpu().numpy(), ref) <= bar(n, half)
        inplace = xd.clone()
        p(inplace, inplace)
        assert rel(inplace.cpu().numpy(), ref) <= bar(n, half)
    r = x.real.copy()
    X = K.ScalarPlan(n, half=half).forward(r)
    assert rel(X, np.fft.fft(r.astype(np.float64))) <= bar(n, half)


@pytest.mark.parametrize("shape", [(262, 2134), (74, 131), (1018, 206)])
def test_bluestein_columns(shape):
    """Two dimensions with Bluestein rows and columns (column tiles of the one-pass
    convolution where they fit, transposes elsewhere)."""
    rng = np.random.default_rng(shape[0])
    for half in (False, True):
        x = data(rng, half, *shape)
        got = K.Cpx2Plan(shape[1], shape[0], half=half)(x)
        assert rel(got, np.fft.fft2(x.astype(np.complex128))) <= bar(x.size, half)


def test_blocking_call_waits_for_null_stream():
    """A buffer the null stream is still producing is complete when a blocking call
    reads it, and blocking and asynchronous calls of one plan keep their order."""
    import torch

    n = 94132
    p = K.CpxPlan(n)
    big = torch.rand(4096, 4096, device="cuda")
    x = torch.zeros(n, 2, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    for _ in range(20):
        big = big @ big * 1e-4
    x[:] = torch.linspace(-1, 1, 2 * n, device="cuda", dtype=torch.float64).view(n, 2)
    got = p(torch.view_as_complex(x))
    ref = np.fft.fft(torch.view_as_complex(x).cpu().numpy())
    assert rel(got.cpu().numpy(), ref) <= bar(n, False)
    xc = torch.view_as_complex(x).clone()
    out = [torch.empty_like(xc) for _ in range(3)]
    st = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    p.run_async(xc, out[0], 1, st[0].cuda_stream)
    p(xc, out[1])
    p.run_async(xc, out[2], 1, st[1].cuda_stream)
    torch.cuda.synchronize()
    for o in out:
        assert rel(o.cpu().numpy(), ref) <= bar(n, False)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n", [128, 512, 2000, 2016, 4096, 4160, 8192, 8320, 16384, 32768,
                               65536, 1 << 18, 1 << 21])
def test_real_rebuild_in_pass(n, half):
    """Half lengths of the compiled row passes: the rebuild in the store, the inverse
    rebuild in the load; a batch with a partial tile, and an inverse whose output
    lies over its own spectra (which takes the separate rebuild)."""
    import torch

    rng = np.random.default_rng(n)
    b = 5
    x = rng.uniform(-1, 1, (b, n)).astype(np.float32 if half else np.float64)
    X = K.ScalarPlan(n, half=half).forward(x)
    assert rel(X, np.fft.rfft(x.astype(np.float64))) <= bar(n, half)
    inv = K.ScalarPlan(n, K.FLAG_INVERSE, half=half)
    ref = 2.0 * x.astype(np.float64)
    assert rel(inv.inverse(X), ref) <= 2 * bar(n, half)
    buf = torch.from_numpy(np.ascontiguousarray(X)).cuda()
    inv.L.kfft_evali_scalar_batch(inv.handle, buf.data_ptr(), buf.data_ptr(), b)
    got = torch.view_as_real(buf).reshape(-1)[:b * n].reshape(b, n)
    assert rel(got.cpu().numpy(), ref) <= 2 * bar(n, half)


# widths: rebuild in the row pass (blocks of four columns, whole and partial), rows
# through Bluestein and rows of two passes (row layout)
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("x", [6, 62, 64, 202, 4160, 74, 16384])
@pytest.mark.parametrize("y", [256, 480, 1000, 2080, 4096, 4160])
def test_column_convolution(y, x, half):
    if x * y > 20e6:
        y = 256
    rng = np.random.default_rng(x * 10000 + y)
    t = np.float32 if half else np.float64
    a, b = (rng.uniform(-1, 1, (y, x)).astype(t) for _ in range(2))
    ref = np.fft.irfft2(np.fft.rfft2(a.astype(np.float64)) * np.fft.rfft2(b.astype(np.float64)),
                        s=(y, x))
    got = K.Conv2Plan(x, y, real=True, half=half)(a, b)
    assert rel(got, 2 * ref) <= 2 * bar(x * y, half)
    raw = K.Conv2Plan(x, y, K.FLAG_DISABLE_NORM, real=True, half=half)(a, b)
    assert rel(raw, ref * (x * y)) <= 2 * bar(x * y, half)


@pytest.mark.parametrize("half,n", [(False, n) for n in (5120, 6144, 6250, 6400, 6561, 7680, 8192)]
                         + [(True, n) for n in (10000, 10240, 15360)])
def test_long_rows_in_one_pass(n, half):
    """Long rows: the one-pass form at its smallest batch (a row per CU) and past it,
    the two-pass form below; forward, normalised inverse, in place."""
    import torch

    rng = np.random.default_rng(n)
    for batch in (255, 256, 259):
        x = data(rng, half, batch, n)
        xd = torch.from_numpy(x).cuda()
        p = K.CpxPlan(n, half=half)
        ref = np.fft.fft(x.astype(np.complex128))
        y = p(xd)
        assert rel(y.cpu().numpy(), ref) <= bar(n, half)
        K.CpxPlan(n, K.FLAG_INVERSE, half=half)(y, y)
        assert rel(y.cpu().numpy(), x) <= 2 * bar(n, half)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n", [257, 1009, 2017, 12289, 65537])
def test_rader_first_value(n, half):
    """X[0] and x[0]: stored and read by the passes themselves out of place, through
    copies in place and where input and output overlap; real input and output."""
    import torch

    rng = np.random.default_rng(n)
    b = 3
    x = data(rng, half, b, n) + 2.0  # (a first value that matters)
    x = x.astype(np.complex64 if half else np.complex128)
    wide = torch.zeros(2 * b * n, dtype=torch.from_numpy(x).dtype, device="cuda")
    ref = np.fft.fft(x.astype(np.complex128))
    p = K.CpxPlan(n, half=half)
    for off in (0, b * n):  # in place, apart in one buffer
        wide[:b * n] = torch.from_numpy(x).cuda().reshape(-1)
        torch.cuda.synchronize()
        p(wide[:b * n].view(b, n), wide[off:off + b * n].view(b, n))
        got = wide[off:off + b * n].view(b, n).cpu().numpy()
        assert rel(got, ref) <= bar(n, half)
        assert rel(got[:, 0], ref[:, 0]) <= bar(n, half)
    r = np.ascontiguousarray(x.real)
    X = K.ScalarPlan(n, half=half).forward(r)
    assert rel(X[:, 0], r.astype(np.float64).sum(axis=1)) <= bar(n, half)
    back = K.ScalarPlan(n, K.FLAG_INVERSE, half=half).inverse(X)
    assert rel(back, r) <= 2 * bar(n, half)
    assert rel(back[:, 0], r[:, 0]) <= 4 * bar(n, half)


def test_column_blocks_of_a_large_matrix():
    """A matrix of more than 256 MiB whose columns run as packed blocks over two
    streams, the last block narrower; forward twice (the scratch in use again)."""
    import torch

    y, x = 8192, 4160
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.view_as_complex(torch.rand(y, x, 2, generator=g, device="cuda") * 2 - 1)
    p, q = K.Cpx2Plan(x, y, half=True), K.Cpx2Plan(x, y, K.FLAG_INVERSE, half=True)
    A = p(a)
    back = q(A)
    assert float((back - a).norm() / a.norm()) <= 2 * bar(x * y, True)
    cols = [0, 1, 1087, 1088, 2175, 3263, 3264, 4159]
    rows = torch.fft.fft(a.cpu().to(torch.complex128), dim=1)[:, cols].numpy()
    ref = np.fft.fft(rows, axis=0)
    assert rel(A[:, cols].cpu().numpy(), ref) <= bar(x * y, True)
    assert torch.equal(torch.view_as_real(p(a)), torch.view_as_real(A))
