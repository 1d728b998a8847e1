"""Benchmark of the batched 1D complex transform on one MI355X.

Workload (the headline configuration): N = 2^16 points, batch 4096, complex,
forward transform, inputs uniform[-1,1) (seeded) resident in HBM before the
timed region.  A step is one batched transform of the whole set through the
C ABI (kfft_eval_cpx_batch_async on the library stream).  Timing uses HIP
events recorded on that stream around exactly K steps.

Forms (all run in one invocation; --form picks the one reported as `value`):
  fp64       the double build (libkfft_amd.so), the plain form
  fp32       the float build (libkfft_amd_half.so): FP32 arithmetic on the
             vector units, FP64-generated twiddles rounded once
  f16, bf16  the precision form: radix-16 stages as split FP16 / BF16 matrix
             products with FP32 accumulation (KFFT_FLAG_GPU_SPLIT_F16 / _BF16)
  f16r, bf16r  the same plus one refinement step on the FP64 residual
             (KFFT_FLAG_GPU_REFINE)
The reported value is GFLOP/s = 5 N log2 N * batch / t.  Every FP32 form
carries its relative L2 error against the FP64 path on two input sets (uniform
noise, and unit noise with 1e-6-amplitude tones); the split forms carry their
matrix-core utilisation (dense FP16/BF16 products issued per second against
the 2.5 PFLOP/s peak).

The CPU baseline is the oracle (a C restatement of the reference's algorithm,
OpenMP over the batch, all host threads) timed on a bounded sample of the same
workload.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
MFMA_PEAK_FLOPS = 2.5e15  # MI355X dense FP16 / BF16 matrix peak
FORMS = ("fp64", "fp32", "f16", "bf16", "f16r", "bf16r")


def _form_flags(form: str) -> int:
    import kfft_amd as K

    f = 0
    if form.startswith("f16"):
        f |= K.FLAG_GPU_SPLIT_F16
    if form.startswith("bf16"):
        f |= K.FLAG_GPU_SPLIT_BF16
    if form.endswith("r"):
        f |= K.FLAG_GPU_REFINE
    return f


def _radix16_stages(describe: str) -> int:
    """Radix-16 stages of a power-of-two plan on the shaped passes: a pass of
    2^a points runs a // 4 radix-16 stages (one fewer when a % 4 == 1)."""
    import re

    m = re.search(r"inner=(\d+) (four-step (\d+)x(\d+)|one-pass)", describe)
    if not m:
        return 0
    lens = [int(m.group(3)), int(m.group(4))] if m.group(3) else [int(m.group(1))]
    total = 0
    for L in lens:
        if L < 16 or L > 4096 or L & (L - 1):
            return 0
        a = L.bit_length() - 1
        q, rr = divmod(a, 4)
        total += q - 1 if (rr == 1 and q > 0) else q
    return total


def _gpu_form(form: str, n: int, batch: int, steps: int, warmup: int, x64, x32, flags: int = 0):
    import torch

    import kfft_amd as K

    half = form != "fp64"
    plan = K.CpxPlan(n, flags | _form_flags(form), half=half)
    x = x32 if half else x64
    y = torch.empty_like(x)
    stream = torch.cuda.ExternalStream(K.load(half).kfft_gpu_stream())
    for _ in range(warmup):
        plan.run_async(x, y, batch)
    K.synchronize(half)
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    wall0 = time.perf_counter()
    t0.record(stream)
    for _ in range(steps):
        plan.run_async(x, y, batch)
    t1.record(stream)
    t1.synchronize()
    wall = time.perf_counter() - wall0
    ms = t0.elapsed_time(t1) / steps
    return plan, y, ms, wall


def _measured_traffic(form: str, n: int, batch: int):
    """HBM bytes of one step from the committed rocprofv3 FETCH_SIZE / WRITE_SIZE
    summary for this workload (profiles/traffic_*.json), or None."""
    path = os.path.join(ROOT, "profiles", f"traffic_c2c_{n}x{batch}.json")
    try:
        with open(path) as f:
            d = json.load(f)
        return d[form]["bytes_per_step"]
    except Exception:
        return None


def ragged_bench(count: int, steps: int, warmup: int, per_item: bool = True):
    """The batching form on the ragged workload: `count` transforms, lengths
    log-uniform over [16, 65536] (15% forced prime, 30% powers of two), half
    complex and half real input, FP32, one persistent launch per batch.  Also
    times the same transforms launched one by one through the batched API."""
    import torch

    import kfft_amd as K
    from kfft_amd.workloads import ragged_batch

    lengths, kinds = ragged_batch(count)
    t0 = time.perf_counter()
    plan = K.RaggedPlan(lengths, kinds, half=True)
    plan_s = time.perf_counter() - t0
    g = torch.Generator(device="cuda").manual_seed(20260105)
    x = torch.rand((plan.in_bytes + 3) // 4, generator=g, device="cuda") * 2 - 1
    y = torch.zeros((plan.out_bytes + 3) // 4, device="cuda")
    torch.cuda.synchronize()
    stream = torch.cuda.ExternalStream(K.load(True).kfft_gpu_stream())
    for _ in range(warmup):
        plan.run_async(x, y)
    K.synchronize(True)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(steps):
        plan.run_async(x, y)
    e1.record(stream)
    e1.synchronize()
    ms = e0.elapsed_time(e1) / steps
    if plan.error():
        raise RuntimeError("ragged batch: a dependency wait timed out")
    # a sample of the batch's outputs against the oracle (outside the timed
    # region): every 1000th transform, each form (power of two, smooth, Rader,
    # Bluestein, real and complex input) among them
    import numpy as np
    import oracle as O

    worst = 0.0
    checked = 0
    xs_h, ys_h = x.cpu().numpy(), y.cpu().numpy()
    for i in range(0, len(lengths), 1000):
        n, k = int(lengths[i]), int(kinds[i])
        a0, b0 = int(plan.in_off[i]) // 4, int(plan.out_off[i]) // 4
        if k == 1:
            xi = xs_h[a0:a0 + n].astype(np.float64)
            ref = O.rfft(xi)
        else:
            xi = xs_h[a0:a0 + 2 * n].view(np.complex64).astype(np.complex128)
            ref = O.fft(xi)
        got = ys_h[b0:b0 + 2 * ref.size].view(np.complex64).astype(np.complex128)
        worst = max(worst, float(np.linalg.norm(got - ref) / np.linalg.norm(ref)))
        checked += 1
    out_len = [(n // 2 + 1) if (k == 1 and n % 2 == 0) else n for n, k in zip(lengths, kinds)]
    alg = float(sum(n * (4 if k == 1 else 8) for n, k in zip(lengths, kinds)) +
                8 * sum(out_len))
    flops = float(sum((2.5 if k == 1 else 5.0) * n * math.log2(n) for n, k in zip(lengths, kinds)))
    res = {"transforms": int(count), "ms_per_batch": round(ms, 4),
           "gflops": round(flops / (ms * 1e-3) / 1e9, 2),
           "achieved_gbs": round(alg / (ms * 1e-3) / 1e9, 1),
           "hbm_frac": round(alg / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
           "alg_bytes": alg, "plan_s": round(plan_s, 2), "plan": plan.describe(),
           "sample_check": {"transforms": checked, "max_rel_l2_vs_oracle": worst,
                            "what": "every 1000th transform of the batch, FP64 oracle on the "
                                    "same float32 inputs"}}
    # shapes ranked by the committed cost model (trained on this GPU's timings)
    model_path = os.path.join(ROOT, "kfft_amd", "data", "cost_model_mi355x.npz")
    if os.path.exists(model_path):
        import numpy as np

        md = np.load(model_path)
        m = K.Mlp(int(md["nin"]), int(md["hidden"]))
        m.set_params(md["params"])
        m.use_as_cost_model()
        try:
            t0 = time.perf_counter()
            tuned = K.RaggedPlan(lengths, kinds, flags=K.FLAG_GPU_TUNED, half=True)
            tplan_s = time.perf_counter() - t0
        finally:
            K.clear_cost_model()
        for _ in range(warmup):
            tuned.run_async(x, y)
        K.synchronize(True)
        e0.record(stream)
        for _ in range(steps):
            tuned.run_async(x, y)
        e1.record(stream)
        e1.synchronize()
        tms = e0.elapsed_time(e1) / steps
        if tuned.error():
            raise RuntimeError("tuned ragged batch: a dependency wait timed out")
        changed = sum(1 for c, d in zip(tuned.classes(), plan.classes()) if c != d)
        res["tuned"] = {"ms_per_batch": round(tms, 4), "speedup_vs_default": round(ms / tms, 3),
                        "plan_s": round(tplan_s, 2), "classes_not_default": changed,
                        "model": "kfft_amd/data/cost_model_mi355x.npz"}
        # the model's picks on the timing database's held-out classes against the
        # exhaustive search over the same choices (measured time per class)
        db_path = os.path.join(ROOT, "kfft_amd", "data", "tune_db_mi355x.npz")
        if os.path.exists(db_path):
            import torch

            from kfft_amd import tune as T

            db = dict(np.load(db_path))
            pred = m.forward(torch.from_numpy(T.features(db).astype(np.float32)).cuda())
            held = T.split(db)
            r = T.regret(db, T.choose(pred.cpu().numpy(), db, held))
            res["tuned"]["regret_vs_exhaustive"] = {
                k: (round(v, 4) if isinstance(v, float) else v) for k, v in r.items()}
            res["tuned"]["regret_vs_exhaustive"]["what"] = (
                "held-out classes of kfft_amd/data/tune_db_mi355x.npz: measured time of the "
                "model's pick / fastest measured choice - 1")
    if per_item:
        # the method without the executor: one asynchronous batched call per transform
        plans = {}
        for n, k in set(zip(lengths.tolist(), kinds.tolist())):
            plans[(n, k)] = K.ScalarPlan(n, half=True) if k == 1 else K.CpxPlan(n, half=True)
        xs = [x[int(o) // 4:] for o in plan.in_off]
        ys = [y[int(o) // 4:] for o in plan.out_off]
        L = K.load(True)

        def one_by_one():
            for i, (n, k) in enumerate(zip(lengths.tolist(), kinds.tolist())):
                p = plans[(n, k)]
                if k == 1:
                    L.kfft_eval_scalar_batch_async(p.handle, xs[i].data_ptr(), ys[i].data_ptr(),
                                                   1, None)
                else:
                    L.kfft_eval_cpx_batch_async(p.handle, xs[i].data_ptr(), ys[i].data_ptr(), 1,
                                                None)
        one_by_one()
        K.synchronize(True)
        e0.record(stream)
        one_by_one()
        e1.record(stream)
        e1.synchronize()
        ms1 = e0.elapsed_time(e1)
        res["one_launch_per_transform_ms"] = round(ms1, 3)
        res["speedup_vs_one_launch_per_transform"] = round(ms1 / ms, 2)
    return res


def _timed(fn, steps: int, warmup: int = 1) -> float:
    """ms per call of a synchronous call sequence, wall clock (host pointers
    are never used: every buffer is device memory)."""
    import torch

    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / steps * 1e3


def _timed_async(plan, x, y, batch, steps, half):
    """ms per batched asynchronous call, HIP events on the library stream."""
    import torch

    import kfft_amd as K

    stream = torch.cuda.ExternalStream(K.load(half).kfft_gpu_stream())
    plan.run_async(x, y, batch)
    K.synchronize(half)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(steps):
        plan.run_async(x, y, batch)
    e1.record(stream)
    e1.synchronize()
    return e0.elapsed_time(e1) / steps


def other_configs(steps: int, only: str = None):
    """The reference's other workloads at their full sizes, plain FP64 unless
    stated: time, algorithmic GB/s against the 8 TB/s roofline, and the
    relative L2 error of a sample against the oracle (or the stated check)."""
    import numpy as np
    import torch

    import kfft_amd as K
    import oracle as O

    out = {}

    def want(name):  # all workloads, or only the named one (profiler runs)
        return only is None or name == only

    def entry(name, ms, alg_bytes, err, **kw):
        gbs = alg_bytes / (ms * 1e-3) / 1e9
        out[name] = dict(ms=round(ms, 4), achieved_gbs=round(gbs, 1),
                         hbm_frac=round(gbs / HBM_PEAK_GBS, 4), rel_err=err, **kw)
        print(f"# config {name}: {ms:.4f} ms, {gbs:.0f} GB/s, err {err:.2e}", file=sys.stderr,
              flush=True)

    def cplx(b, n, dt=torch.complex128, seed=1):
        g = torch.Generator(device="cuda").manual_seed(seed)
        rt = torch.float64 if dt == torch.complex128 else torch.float32
        return torch.view_as_complex(torch.rand(b, n, 2, generator=g, device="cuda", dtype=rt)
                                     * 2 - 1).contiguous()

    def rel(a, b):
        return float(np.linalg.norm(a - b) / np.linalg.norm(b))

    # 4096 x 256 FP64: forward, then inverse with DISABLE_NORM (checked as inverse / N)
    if want("c2c_4096x256_fwd_inv_f64"):
        # the 16 MiB set fits the caches: timed over 24 rotating buffer sets
        # (768 MiB, past the 256 MB Infinity Cache) so that it comes from HBM,
        # and also in one set (cache resident) for comparison
        n, b, R = 4096, 256, 24
        xs = [cplx(b, n, seed=100 + i) for i in range(R)]
        ys = [torch.empty_like(xs[0]) for _ in range(R)]
        zs = [torch.empty_like(xs[0]) for _ in range(R)]
        fw, iv = K.CpxPlan(n), K.CpxPlan(n, K.FLAG_INVERSE | K.FLAG_DISABLE_NORM)
        stream = torch.cuda.ExternalStream(K.load(False).kfft_gpu_stream())

        def rotating(p, src, dst, reps):
            for i in range(R):
                p.run_async(src[i], dst[i], b)
            K.synchronize(False)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for j in range(reps):
                for i in range(R):
                    p.run_async(src[i], dst[i], b)
            e1.record(stream)
            e1.synchronize()
            return e0.elapsed_time(e1) / (reps * R)
        tf = rotating(fw, xs, ys, max(2, steps // 2))
        ti = rotating(iv, ys, zs, max(2, steps // 2))
        tfc = _timed_async(fw, xs[0], ys[0], b, steps * 10, False)
        tic = _timed_async(iv, ys[0], zs[0], b, steps * 10, False)
        x, y, z = xs[0], ys[0], zs[0]
        err = max(rel(y[:2].cpu().numpy(), O.fft(x[:2].cpu().numpy())),
                  rel((z / n).cpu().numpy(), x.cpu().numpy()))
        xh = x.cpu().numpy()
        ofw, oiv = O.Plan(n), O.Plan(n, O.FLAG_INVERSE | O.FLAG_DISABLE_NORM)
        cpu = _cpu_ms(lambda v, t: oiv(ofw(v, t), t), xh, 1.0)
        entry("c2c_4096x256_fwd_inv_f64", tf + ti, 2 * 2.0 * n * 16 * b, err,
              fwd_ms=round(tf, 4), inv_ms=round(ti, 4), buffers="24 rotating sets (768 MiB)",
              cache_resident_ms=round(tfc + tic, 4), **cpu)
        del xs, ys, zs, x, y, z
    # hard lengths, ~256 MB per set
    for n, b in [(1000, 16384), (6561, 2560), (1009, 16384), (65537, 256), (1 << 20, 16)]:
        if not want(f"c2c_{n}x{b}_f64"):
            continue
        x = cplx(b, n)
        y = torch.empty_like(x)
        p = K.CpxPlan(n)
        ms = _timed_async(p, x, y, b, steps, False)
        err = rel(y[0].cpu().numpy(), O.fft(x[0].cpu().numpy()))
        sb = max(2, min(b, (1 << 22) // n))  # a sample of about 4M points
        op = O.Plan(n)
        cpu = _cpu_ms(lambda v, t: op(v, t), x[:sb].cpu().numpy(), b / sb)
        entry(f"c2c_{n}x{b}_f64", ms, 2.0 * n * 16 * b, err, plan=p.describe(),
              cpu_sample=f"{sb} of {b} transforms", **cpu)
        del x, y
    # real input 2^18 x 512
    if want("r2c_262144x512_f64"):
        n, b = 1 << 18, 512
        g = torch.Generator(device="cuda").manual_seed(2)
        xr = torch.rand(b, n, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        sp = K.ScalarPlan(n)
        yr = torch.empty(b, n // 2 + 1, dtype=torch.complex128, device="cuda")
        L = K.load(False)
        ms = _timed(lambda: L.kfft_eval_scalar_batch(sp.handle, xr.data_ptr(), yr.data_ptr(), b),
                    steps)
        err = rel(yr[0].cpu().numpy(), O.rfft(xr[0].cpu().numpy()))
        sb = 16
        op = O.ScalarPlan(n)
        cpu = _cpu_ms(lambda v, t: op.forward(v, threads=t), xr[:sb].cpu().numpy(), b / sb)
        entry("r2c_262144x512_f64", ms, b * (n * 8.0 + (n // 2 + 1) * 16.0), err,
              cpu_sample=f"{sb} of {b} transforms", **cpu)
        del xr, yr
    # 2D 8192 x 8192 complex FP32, forward and inverse (plain FP32 and split FP16)
    for tag, fl in (("f32", 0), ("f32_split_f16", K.FLAG_GPU_SPLIT_F16)):
        if not want(f"c2c_2d_8192x8192_{tag}"):
            continue
        n = 8192
        a = cplx(n, n, torch.complex64, seed=3)
        f2 = K.Cpx2Plan(n, n, fl, half=True)
        i2 = K.Cpx2Plan(n, n, fl | K.FLAG_INVERSE, half=True)
        A = torch.empty_like(a)
        B = torch.empty_like(a)
        L32 = K.load(True)
        tf = _timed(lambda: L32.kfft_eval2_cpx(f2.handle, a.data_ptr(), A.data_ptr()), steps)
        ti = _timed(lambda: L32.kfft_eval2_cpx(i2.handle, A.data_ptr(), B.data_ptr()), steps)
        err = rel(B.to(torch.complex128).cpu().numpy(), a.to(torch.complex128).cpu().numpy())
        # CPU: 2 directions x (8192 row + 8192 column transforms of 8192 points),
        # from a sample of 256 row transforms in FP64
        sb = 256
        op = O.Plan(n)
        cpu = _cpu_ms(lambda v, t: op(v, t), a[:sb].to(torch.complex128).cpu().numpy(),
                      2 * 2 * n / sb)
        entry(f"c2c_2d_8192x8192_{tag}", tf + ti, 2 * 2.0 * n * n * 8, err, fwd_ms=round(tf, 4),
              inv_ms=round(ti, 4), check="inverse(forward(x)) against x",
              cpu_sample="256 FP64 row transforms of 8192 points, scaled to 4 x 8192",
              **cpu)
        del a, A, B
    # real 2D convolution: 4096^2 image (uniform[0,1)) with a 63^2 Gaussian plus noise kernel,
    # both zero-padded to 4160^2; the reference's even-y quirk makes the output 2x the
    # circular convolution.  Checked against an FP64 direct sum on a 64 x 64 crop.
    if not any(want(f"conv2d_real_4160x4160_{t}") for t in ("f32", "f32_split_f16", "f64")):
        return out
    N, M, k = 4160, 4096, 63
    rng = np.random.default_rng(4)
    img = np.zeros((N, N))
    img[:M, :M] = rng.uniform(0, 1, (M, M))
    yy, xx = np.mgrid[:k, :k] - k // 2
    ker = np.exp(-(xx ** 2 + yy ** 2) / (2 * 10.0 ** 2)) + 0.01 * rng.uniform(-1, 1, (k, k))
    kp = np.zeros((N, N))
    kp[:k, :k] = ker
    r0, c0 = 1000, 2000
    crop = np.zeros((64, 64))
    win = img[r0 - k + 1:r0 + 64, c0 - k + 1:c0 + 64]
    for dy in range(k):
        for dx in range(k):
            crop += ker[dy, dx] * win[k - 1 - dy:k - 1 - dy + 64, k - 1 - dx:k - 1 - dx + 64]
    for tag, half, fl in (("f32", True, 0), ("f32_split_f16", True, K.FLAG_GPU_SPLIT_F16),
                          ("f64", False, 0)):
        if not want(f"conv2d_real_4160x4160_{tag}"):
            continue
        dt = torch.float32 if half else torch.float64
        ia = torch.from_numpy(img).to(dt).cuda()
        ka = torch.from_numpy(kp).to(dt).cuda()
        o = torch.empty_like(ia)
        cp = K.Conv2Plan(N, N, fl, real=True, half=half)
        Lh = K.load(half)
        ms = _timed(lambda: Lh.kfft_eval2_conv_scalar(cp.handle, ia.data_ptr(), ka.data_ptr(),
                                                      o.data_ptr()), steps)
        got = o[r0:r0 + 64, c0:c0 + 64].to(torch.float64).cpu().numpy() / 2.0
        # CPU: three 2D transforms of 4160 x 4160 (rows and columns) plus the
        # product, from a sample of 256 FP64 complex transforms of 4160 points
        sb = 256
        op = O.Plan(N)
        cpu = _cpu_ms(lambda v, t: op(v, t), (img[:sb] + 0j).astype(np.complex128),
                      3 * 2 * N / sb)
        entry(f"conv2d_real_4160x4160_{tag}", ms, 3.0 * N * N * (4 if half else 8),
              rel(got, crop), check="64x64 crop against an FP64 direct sum (output / 2)",
              cpu_sample="256 FP64 complex transforms of 4160 points, scaled to 3 x 2 x 4160",
              **cpu)
        del ia, ka, o
    return out


def cpu_threads() -> int:
    """Threads for the CPU baselines: the CPU share this process is given
    (OMP_NUM_THREADS when set, which the GPU hosts set to the cores allotted per
    GPU), else every core in the process's affinity set."""
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit() and int(env) > 0:
        return int(env)
    try:
        return len(os.sched_getaffinity(0))
    except Exception:
        return os.cpu_count() or 1


def _median_time(fn, seconds: float, min_runs: int = 3):
    times = []
    t_all = time.perf_counter()
    while len(times) < min_runs or time.perf_counter() - t_all < seconds:
        t = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t)
    return sorted(times)[len(times) // 2], len(times), time.perf_counter() - t_all


def cpu_baseline(n: int, sample_batch: int, seconds: float = 10.0):
    """The oracle (C restatement of the reference's double build, OpenMP over the
    batch) on a bounded sample of the headline workload: all allotted threads,
    and one thread on a smaller sample."""
    import numpy as np

    import oracle as O

    rng = np.random.default_rng(7)
    x = rng.uniform(-1, 1, (sample_batch, n)) + 1j * rng.uniform(-1, 1, (sample_batch, n))
    threads = cpu_threads()
    p = O.Plan(n)
    p(x[:1], threads=threads)  # warm
    med, runs, total = _median_time(lambda: p(x, threads=threads), seconds)
    gflops = 5 * n * math.log2(n) * sample_batch / med / 1e9
    one = x[:max(1, sample_batch // 16)]
    med1, runs1, total1 = _median_time(lambda: p(one, threads=1), seconds / 4)
    gflops1 = 5 * n * math.log2(n) * len(one) / med1 / 1e9
    try:
        affinity = len(os.sched_getaffinity(0))
    except Exception:
        affinity = None
    return {"value": round(gflops, 3), "unit": "GFLOP/s", "cores": threads, "kind": "port",
            "sample": f"oracle FP64 C2C N={n} x {sample_batch} transforms, median of "
                      f"{runs} passes ({med:.3f} s each, {total:.1f} s in all), OpenMP over the "
                      f"batch on {threads} threads",
            "single_thread": {"value": round(gflops1, 3), "unit": "GFLOP/s",
                              "sample": f"N={n} x {len(one)} transforms, median of {runs1} passes "
                                        f"({med1:.3f} s each)"},
            "host": {"os_cpu_count": os.cpu_count(), "affinity_cpus": affinity,
                     "omp_num_threads": os.environ.get("OMP_NUM_THREADS")}}


def _cpu_ms(plan_fn, x, scale: float, seconds: float = 1.5) -> dict:
    """Oracle time of one bounded sample (all allotted threads), scaled to the
    full workload by `scale`."""
    threads = cpu_threads()
    plan_fn(x[:1], threads)
    med, runs, _ = _median_time(lambda: plan_fn(x, threads), seconds)
    return {"cpu_ms": round(med * scale * 1e3, 3), "cpu_threads": threads,
            "cpu_sample_ms": round(med * 1e3, 3), "cpu_scale": round(scale, 3)}


def copy_reference_gbs(gib: int = 2) -> float:
    """Read + write GB/s of a plain device-to-device copy of `gib` GiB (torch's
    copy kernel): what a data-movement kernel reaches on this GPU."""
    import torch

    a = torch.empty(gib << 27, dtype=torch.complex64, device="cuda")
    b = torch.empty_like(a)
    for _ in range(2):
        b.copy_(a)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(5):
        b.copy_(a)
    e1.record()
    e1.synchronize()
    ms = e0.elapsed_time(e1) / 5
    del a, b
    return round(2 * (gib << 30) / (ms * 1e-3) / 1e9, 1)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--n", type=int, default=1 << 16)
    ap.add_argument("--batch", type=int, default=4096)
    ap.add_argument("--form", choices=list(FORMS), default="f16")
    ap.add_argument("--forms", default=",".join(FORMS),
                    help="comma-separated forms to run (the reported one is always included)")
    ap.add_argument("--only", action="store_true",
                    help="time the reported form alone (no accuracy sets, no ragged batch, no "
                         "CPU baseline): for profiler runs")
    ap.add_argument("--cpu-sample", type=int, default=512)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--ragged", type=int, default=20000,
                    help="transforms of the ragged batching-form workload (0: skip)")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the reference's other workloads (4096x256, hard lengths, real "
                         "2^18, 2D 8192^2, real conv2d 4160^2)")
    ap.add_argument("--onchip", action="store_true",
                    help="plan with KFFT_FLAG_GPU_ONCHIP (fused persistent two-pass kernel)")
    ap.add_argument("--config", default=None,
                    help="time one of the reference's other workloads alone (a key of the "
                         "'configs' object, e.g. c2c_1000x16384_f64) and print its entry: for "
                         "profiler runs")
    ap.add_argument("--copy-ref", action="store_true",
                    help="after timing, run one plain device copy of the FP64 input (4 GiB at the "
                         "default size) so that profiler byte counters can be calibrated")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this benchmark runs on one GPU; the batch shards across GPUs "
                          "with no exchange, but multi-GPU runs are not part of it",
                          "n_gpus": args.gpus}))
        sys.exit(2)

    import numpy as np
    import torch

    if args.config:
        res = other_configs(max(1, args.steps), only=args.config)
        if args.config not in res:
            print(json.dumps({"error": f"unknown workload {args.config}"}))
            sys.exit(2)
        print(json.dumps({"config": args.config, **res[args.config]}))
        return
    n, batch = args.n, args.batch
    forms = [f for f in FORMS if f in args.forms.split(",") or f in (args.form, "fp64")]
    if args.only:
        forms = [args.form]
        args.ragged, args.no_cpu = 0, True
    g = torch.Generator(device="cuda").manual_seed(20260103)
    # set A: uniform[-1,1) re/im, rounded to FP32 once so that every form sees the same values
    x32 = torch.view_as_complex(
        torch.rand(batch, n, 2, generator=g, device="cuda", dtype=torch.float32) * 2 - 1
    ).contiguous()
    x64 = x32.to(torch.complex128)

    import kfft_amd as K

    flags = K.FLAG_GPU_ONCHIP if args.onchip else 0
    res = {}
    for form in forms:
        plan, y, ms, wall = _gpu_form(form, n, batch, args.steps, args.warmup, x64, x32, flags)
        if plan.error():
            raise RuntimeError(f"{form}: the fused transform reported a failed dependency wait")
        res[form] = {"plan": plan, "ms": ms, "y": y}
        print(f"# {form}: {ms:.4f} ms/step ({plan.describe()})", file=sys.stderr, flush=True)

    def rel_err(y, ref):
        return (torch.linalg.vector_norm(y.to(torch.complex128) - ref) /
                torch.linalg.vector_norm(ref)).item()

    # the on-chip form (single pass by workgroup pairs) of the FP32 forms
    if not args.onchip and not args.only:
        for form in ("fp32", "f16"):
            if form in res:
                p, _, oms, _ = _gpu_form(form, n, batch, args.steps, args.warmup, x64, x32,
                                         K.FLAG_GPU_ONCHIP)
                if p.error():
                    raise RuntimeError(f"{form} on-chip: a dependency wait timed out")
                res[form]["onchip_ms"] = oms
                print(f"# {form} on-chip: {oms:.4f} ms/step ({p.describe()})", file=sys.stderr,
                      flush=True)
                del p, _

    # accuracy on set A against the FP64 path
    y64 = res["fp64"]["y"] if "fp64" in res else None
    for form in forms:
        if form != "fp64" and y64 is not None:
            res[form]["err_uniform"] = rel_err(res[form]["y"], y64)
        del res[form]["y"]
    del y64
    if args.copy_ref:
        # one plain device copy of the FP64 input (4 GiB at the default size): the
        # reference for calibrating profiler byte counters
        ref = torch.empty_like(x64)
        ref.copy_(x64)
        torch.cuda.synchronize()
        copy_ref_bytes = 2 * x64.numel() * x64.element_size()
        del ref
    # set B: unit noise plus five 1e-6-amplitude tones per transform
    if not args.only:
        t = torch.arange(n, device="cuda", dtype=torch.float64)
        freqs = torch.randint(0, n, (batch, 5), generator=g, device="cuda")
        xb = x64.clone()
        for j in range(5):
            ph = 2 * math.pi * (freqs[:, j:j + 1].to(torch.float64) * t[None, :] % n) / n
            xb += 1e-6 * torch.polar(torch.ones_like(ph), ph)
        xb32 = xb.to(torch.complex64)
        xb = xb32.to(torch.complex128)
        del t, freqs
        torch.cuda.synchronize()
        yb64 = torch.empty_like(xb)
        K.CpxPlan(n, 0)(xb, out=yb64)
        yb = torch.empty_like(xb32)
        for form in forms:
            if form != "fp64":
                K.CpxPlan(n, _form_flags(form), half=True)(xb32, out=yb)
                res[form]["err_tones"] = rel_err(yb, yb64)
        del yb, yb64, xb, xb32
    del x64

    form = args.form
    plan, ms = res[form]["plan"], res[form]["ms"]
    esz = 8 if form != "fp64" else 16
    flops = 5.0 * n * math.log2(n) * batch
    value = flops / (ms * 1e-3) / 1e9
    alg_bytes = 2.0 * n * esz * batch
    achieved = alg_bytes / (ms * 1e-3) / 1e9
    r16 = _radix16_stages(res["fp32"]["plan"].describe()) if "fp32" in res else 0

    def form_entry(f, r):
        e = {"ms_per_step": round(r["ms"], 4),
             "gflops": round(flops / (r["ms"] * 1e-3) / 1e9, 2),
             "hbm_frac": round(2.0 * n * (8 if f != "fp64" else 16) * batch /
                               (r["ms"] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
             "speedup_vs_fp64": round(res["fp64"]["ms"] / r["ms"], 3) if "fp64" in res else None}
        if "err_uniform" in r:
            e["rel_l2_vs_fp64"] = {"uniform": r["err_uniform"], "tones_1e-6": r["err_tones"]}
        if "onchip_ms" in r:
            e["onchip"] = {"ms_per_step": round(r["onchip_ms"], 4),
                           "hbm_frac": round(2.0 * n * 8 * batch / (r["onchip_ms"] * 1e-3) / 1e9 /
                                             HBM_PEAK_GBS, 4),
                           "form": "single pass by workgroup pairs (KFFT_FLAG_GPU_ONCHIP)"}
        if f[:3] in ("f16", "bf1"):
            # per 64 butterflies: 2 groups x (3 products (F16) or 6 (BF16)) x 2 halves (Re, Im)
            per_wave = 12 if f.startswith("f16") else 24
            mf = r16 * (n // 16 // 64) * per_wave * (32 * 32 * 16 * 2) * batch
            passes = 2 if f.endswith("r") else 1
            e["mfma"] = {"flop_per_step": mf * passes,
                         "util": round(mf * passes / (r["ms"] * 1e-3) / MFMA_PEAK_FLOPS, 4),
                         "radix16_stages": r16}
        return e

    out = {
        "metric": "batched C2C GFLOP/s (5N*log2N/t) & %HBM peak, FP32-split vs FP64 at <=1e-6",
        "value": round(value, 2),
        "unit": "GFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32" if form != "fp64" else "f64",
        "data": "synthetic uniform[-1,1) seeded, resident in HBM",
        "config": {"workload": f"batched 1D C2C forward N={n} batch={batch}", "n": n,
                   "batch": batch, "form": form, "plan": plan.describe(),
                   "onchip": bool(args.onchip)},
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": None,
                     "kernel": "whole transform (all passes of one step)",
                     "alg_bytes_per_step": alg_bytes},
        "forms": {f: form_entry(f, r) for f, r in res.items()},
    }
    if args.copy_ref:
        out["copy_ref_bytes"] = copy_ref_bytes
    if not args.only:
        # what a plain copy reaches here: the practical ceiling of a kernel that
        # reads and writes the data once
        out["roofline"]["copy_ref_gbs"] = copy_reference_gbs()
    if not args.no_configs and not args.only:
        out["configs"] = other_configs(max(2, args.steps // 4))
    if args.ragged:
        out["ragged"] = ragged_bench(args.ragged, max(3, args.steps // 2), 1)
        print(f"# ragged: {out['ragged']['ms_per_batch']} ms per batch", file=sys.stderr, flush=True)
    traffic = None if args.onchip else _measured_traffic(form, n, batch)
    if traffic is not None:
        out["roofline"]["traffic"] = traffic
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(n, args.cpu_sample)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
