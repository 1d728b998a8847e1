"""Performance cases of the transform engine: what its users have it compute.

listed() holds the fixed cases, draw() gives more of the same ranges.  A case is
a plain dict; its "kind" says which entry point carries it:

  single   one transform per call through the blocking entry point
  batch    many transforms of one length on device buffers, asynchronous
  real     batched real input: forward, then the inverse of its spectrum
  image    2D complex transform: forward, then the inverse of its spectrum
  conv2d   real 2D circular convolution of two images
  ragged   uneven lengths, complex and real, in one call

"type" is f64 (the double library), f32 (the float library) or f16 (the float
library's split matrix-core form, FP32 in and out).  prepare() makes the seeded
inputs, the plan and the output buffers on the GPU, run() makes one pass, work()
is the data and arithmetic a pass cannot do without, exact() the FP64 result.
"""
import concurrent.futures
import math

import numpy as np
import torch

import kfft_amd as K
from kfft_amd import workloads

MAX_POINTS = {"f64": 1 << 24, "f32": 1 << 25, "f16": 1 << 25}


def listed():
    return [
        # one short signal at a time: call and launch latency
        dict(name="single_1024_f64", kind="single", n=1024, type="f64"),
        # one long signal of an awkward length (2^2 101 233): a chirp convolution
        dict(name="single_94132_f64", kind="single", n=94132, type="f64"),
        # a small batch of frames, to the spectrum and back (filtering loops)
        dict(name="batch_4096x256_f64_round", kind="batch", n=4096, batch=256, type="f64",
             direction="both"),
        # the hard lengths at about 256 MB a set: an odd prime power, a short and a
        # long prime, and a long power of two with few transforms
        dict(name="batch_6561x2560_f64", kind="batch", n=6561, batch=2560, type="f64",
             direction="forward"),
        dict(name="batch_1009x16384_f64", kind="batch", n=1009, batch=16384, type="f64",
             direction="forward"),
        dict(name="batch_65537x256_f64", kind="batch", n=65537, batch=256, type="f64",
             direction="forward"),
        dict(name="batch_2p20x16_f64", kind="batch", n=1 << 20, batch=16, type="f64",
             direction="forward"),
        # real signals, spectrum and back (two directions of the half-length form)
        dict(name="real_2p18x512_f64_round", kind="real", n=1 << 18, batch=512, type="f64"),
        # the largest: the throughput workload in the split matrix-core form
        dict(name="batch_2p16x4096_f16", kind="batch", n=1 << 16, batch=4096, type="f16",
             direction="forward"),
        # a large image, to the spectrum and back
        dict(name="image_8192x8192_f32_round", kind="image", x=8192, y=8192, type="f32"),
        # a 4096^2 image filtered by a 63^2 kernel, zero-padded to 4160^2
        dict(name="conv2d_4160x4160_f32", kind="conv2d", x=4160, y=4160, taps=63, type="f32"),
        # mixed traffic: 20,000 signals of uneven lengths, half of them real
        dict(name="ragged_20000_f32", kind="ragged", count=20000, hi=65536, lengths_seed=20260104,
             type="f32"),
    ]


# ----------------------------------------------------------------------- drawing
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_near(n, primes=(2, 3, 5, 7)):
    """The smallest number from n on with no prime factor outside `primes`."""
    while True:
        m = n
        for p in primes:
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


def _length(rng, lo, hi):
    """A length of [lo, hi], log-uniform: powers of two, smooth lengths and any."""
    n = _log_int(rng, lo, hi)
    how = rng.random()
    if how < 0.35:
        return 1 << int(round(math.log2(n)))
    if how < 0.65:
        return min(_smooth_near(n), hi)
    return n


def draw(rng):
    kind = rng.choice(["single", "batch", "batch", "batch", "real", "image", "conv2d", "ragged"])
    kind_type = rng.choice(["f64", "f32"])
    if kind == "single":
        return dict(kind=kind, n=_length(rng, 16, 1 << 17), type=kind_type)
    if kind in ("batch", "real"):
        if kind == "batch" and rng.random() < 0.2:
            kind_type = "f16"
            n = 1 << rng.randint(8, 18)
        else:
            n = _length(rng, 16, 1 << (20 if kind == "batch" else 18))
        top = MAX_POINTS[kind_type]
        if kind == "real":
            top *= 2
        points = _log_int(rng, max(2 * n, 1 << 18), top)
        case = dict(kind=kind, n=n, batch=max(1, points // n), type=kind_type)
        if kind == "batch":
            case["direction"] = rng.choice(["forward", "both"])
        return case
    if kind == "image":
        return dict(kind=kind, x=_smooth_near(_log_int(rng, 128, 4096)),
                    y=_smooth_near(_log_int(rng, 128, 4096)), type=kind_type)
    if kind == "conv2d":
        return dict(kind=kind, x=_smooth_near(_log_int(rng, 64, 2048), (2, 3, 5, 13)) * 2,
                    y=_smooth_near(_log_int(rng, 64, 2048), (2, 3, 5, 13)) * 2,
                    taps=2 * rng.randint(1, 31) + 1, type=kind_type)
    return dict(kind=kind, count=_log_int(rng, 200, 8000), hi=_log_int(rng, 2048, 65536),
                lengths_seed=rng.randrange(1 << 30), type="f32")


# ------------------------------------------------------------------------- inputs
def _real_type(case):
    return torch.float64 if case["type"] == "f64" else torch.float32


def _complex_type(case):
    return torch.complex128 if case["type"] == "f64" else torch.complex64


def _uniform(case, seed, *shape, low=-1.0):
    """Seeded uniform [low, 1) reals on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = torch.rand(*shape, generator=g, device="cuda", dtype=_real_type(case))
    return r if low == 0.0 else r.mul_(1.0 - low).add_(low)


def _uniform_complex(case, seed, *shape):
    return torch.view_as_complex(_uniform(case, seed, *shape, 2))


def _ragged_lengths(case):
    return workloads.ragged_batch(case["count"], case["lengths_seed"], hi=case["hi"])


def _inputs(case, seed):
    """The input tensors of one pass, on the GPU."""
    kind = case["kind"]
    if kind == "single":
        return [_uniform_complex(case, seed, case["n"])]
    if kind == "batch":
        return [_uniform_complex(case, seed, case["batch"], case["n"])]
    if kind == "real":
        return [_uniform(case, seed, case["batch"], case["n"])]
    if kind == "image":
        return [_uniform_complex(case, seed, case["y"], case["x"])]
    if kind == "conv2d":
        # an image in [0, 1) and a Gaussian kernel with noise, both zero-padded
        y, x = case["y"], case["x"]
        t = min(case["taps"], x, y)
        image = torch.zeros(y, x, dtype=_real_type(case), device="cuda")
        image[:y - t, :x - t] = _uniform(case, seed, y - t, x - t, low=0.0)
        at = torch.arange(t, device="cuda", dtype=_real_type(case)) - t // 2
        bell = torch.exp(-at ** 2 / 200.0)
        kernel = torch.zeros_like(image)
        kernel[:t, :t] = bell[:, None] * bell + 0.01 * _uniform(case, seed + 1, t, t)
        return [image, kernel]
    raise ValueError(kind)


def prepare(case, seed):
    kind, half = case["kind"], case["type"] != "f64"
    flags = K.FLAG_GPU_SPLIT_F16 if case["type"] == "f16" else 0
    state = dict(kind=kind)
    if kind == "ragged":
        lengths, kinds = _ragged_lengths(case)
        state["plan"] = K.RaggedPlan(lengths, kinds, half=half)
        state["in"] = _uniform(case, seed, state["plan"].in_bytes // 4)
        state["out"] = torch.zeros(state["plan"].out_bytes // 4, device="cuda")
        return state
    state["in"] = _inputs(case, seed)
    x = state["in"][0]
    if kind in ("single", "batch"):
        state["plan"] = K.CpxPlan(case["n"], flags, half=half)
        state["out"] = torch.empty_like(x)
        state["batch"] = case.get("batch", 1)
        if case.get("direction") == "both":
            state["inverse"] = K.CpxPlan(case["n"], flags | K.FLAG_INVERSE, half=half)
            state["back"] = torch.empty_like(x)
    elif kind == "real":
        state["plan"] = K.ScalarPlan(case["n"], half=half)
        state["inverse"] = K.ScalarPlan(case["n"], K.FLAG_INVERSE, half=half)
        state["batch"] = case["batch"]
        state["out"] = torch.empty(case["batch"], state["plan"].out_len, device="cuda",
                                   dtype=_complex_type(case))
        state["back"] = torch.empty_like(x)
    elif kind == "image":
        state["plan"] = K.Cpx2Plan(case["x"], case["y"], half=half)
        state["inverse"] = K.Cpx2Plan(case["x"], case["y"], K.FLAG_INVERSE, half=half)
        state["out"], state["back"] = torch.empty_like(x), torch.empty_like(x)
    else:
        state["plan"] = K.Conv2Plan(case["x"], case["y"], real=True, half=half)
        state["out"] = torch.empty_like(x)
    return state


# --------------------------------------------------------------------------- a pass
def run(state):
    kind, plan, out = state["kind"], state["plan"], state["out"]
    if kind == "ragged":
        plan.run_async(state["in"], out)
        return out
    if kind == "single":
        return plan(state["in"][0], out)
    if kind == "conv2d":
        return plan(state["in"][0], state["in"][1], out)
    if kind == "image":
        plan(state["in"][0], out)
        return out, state["inverse"](out, state["back"])
    plan.run_async(state["in"][0], out, state["batch"])
    if "inverse" not in state:
        return out
    state["inverse"].run_async(out, state["back"], state["batch"])
    return out, state["back"]


# ------------------------------------------------------------------ work and results
def work(case):
    """Each direction reads its input once and writes its output once; 5 N log2 N
    operations per complex transform of N points, half of it for a real one."""
    kind, real = case["kind"], 8 if case["type"] == "f64" else 4
    if kind == "ragged":
        lengths, kinds = _ragged_lengths(case)
        n, k = lengths.astype(np.float64), kinds.astype(bool)
        bins = np.where(k & (lengths % 2 == 0), lengths // 2 + 1, lengths)
        return dict(bytes=float((n * real * np.where(k, 1, 2) + bins * 2.0 * real).sum()),
                    flops=float((n * np.log2(n) * np.where(k, 2.5, 5.0)).sum()))
    if kind in ("single", "batch"):
        n, both = case["n"], 2 if case.get("direction") == "both" else 1
        batch = case.get("batch", 1)
        return dict(bytes=4.0 * real * n * batch * both,
                    flops=5.0 * n * math.log2(n) * batch * both)
    if kind == "real":
        n, batch = case["n"], case["batch"]
        bins = n // 2 + 1 if n % 2 == 0 else n
        return dict(bytes=2.0 * real * batch * (n + 2 * bins),
                    flops=2 * 2.5 * n * math.log2(n) * batch)
    points = case["x"] * case["y"]
    if kind == "image":
        return dict(bytes=2 * 4.0 * real * points, flops=2 * 5.0 * points * math.log2(points))
    # three real transforms of the image size and a product over half the spectrum
    return dict(bytes=3.0 * real * points, flops=3 * 2.5 * points * math.log2(points) + 3.0 * points)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ragged":
        return _exact_ragged(case, seed)
    given = [t.to(torch.complex128 if t.is_complex() else torch.float64).cpu()
             for t in _inputs(case, seed)]
    x = given[0]
    if kind == "single":
        return torch.fft.fft(x)
    if kind == "batch":
        spectrum = torch.fft.fft(x)
        return (spectrum, x) if case["direction"] == "both" else spectrum
    if kind == "real":
        # an even length's inverse is the library's documented twice the signal
        if case["n"] % 2 == 0:
            return torch.fft.rfft(x), 2 * x
        return torch.fft.fft(x), x
    if kind == "image":
        return torch.fft.fft2(x), x
    # as the real inverse: twice the circular convolution for an even width
    return 2 * torch.fft.irfft2(torch.fft.rfft2(x) * torch.fft.rfft2(given[1]), s=x.shape)


def _exact_ragged(case, seed):
    lengths, kinds = _ragged_lengths(case)
    in_off, out_off, in_bytes, out_bytes = _packed(lengths, kinds)
    x = _uniform(case, seed, in_bytes // 4).cpu().numpy().astype(np.float64)
    y = np.zeros(out_bytes // 4)

    def one(i):
        n, a, b = int(lengths[i]), in_off[i] // 4, out_off[i] // 4
        if kinds[i] == K.RAGGED_REAL:
            z = (np.fft.rfft if n % 2 == 0 else np.fft.fft)(x[a:a + n])
        else:
            z = np.fft.fft(x[a:a + 2 * n].view(np.complex128))
        y[b:b + 2 * z.size] = z.view(np.float64)

    with concurrent.futures.ThreadPoolExecutor(8) as pool:
        list(pool.map(one, range(len(lengths)), chunksize=64))
    return torch.from_numpy(y)


def _packed(lengths, kinds):
    """The packed layout of FP32 ragged batches: transforms in order, each starting
    on a 256-byte boundary."""
    def place(sizes):
        starts, at = [], 0
        for s in sizes:
            at = (at + 255) // 256 * 256
            starts.append(at)
            at += s
        return starts, at
    ins, outs = [], []
    for n, k in zip(lengths.tolist(), kinds.tolist()):
        real = k == K.RAGGED_REAL
        ins.append(n * (4 if real else 8))
        outs.append(8 * (n // 2 + 1 if real and n % 2 == 0 else n))
    in_off, in_bytes = place(ins)
    out_off, out_bytes = place(outs)
    return in_off, out_off, in_bytes, out_bytes
