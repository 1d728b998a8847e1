// C-ABI of the MI355X transform engine: the reference's kfft.h entry points
// (complex, scalar, 2D, conv, conv2d, service, pool) plus the additive
// batched / asynchronous / device-memory entry points of kfft_gpu.h.
//
// Compiled twice: once with kfft_scalar = double (libkfft_amd.so) and once
// with KFFT_HALF_SCALAR, kfft_scalar = float (libkfft_amd_half.so), exactly as
// the reference selects its precision at build time (incs/kfft_types.h:21-25).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <new>

#include "../../include/kfft.h"
#include "../../include/kfft_simd_check.h"
#include "kfa_engine.h"
#include "kfa_kernels.h"
#include "kfa_mlp.h"

#include <map>

using namespace kfa;

static const int PREC = (int)sizeof(kfft_scalar);
static const size_t CPXB = sizeof(kfft_cpx);

// ============================================================ GPU objects
// Device-side state of a plan.  Objects are registered with the pool that
// holds the plan and destroyed when that pool is freed or cleared.
struct GpuObj {
    GpuObj* next = nullptr;
    std::mutex mu;   // one evaluation of a plan at a time (scratch is shared)
    DevBuf scratch;  // engine scratch
    DevBuf stage_in, stage_in2, stage_out; // host-pointer staging
    DevBuf work_a, work_b; // plan-level work buffers (convolution, 2D)
    // completion of the plan's last enqueued evaluation, on whatever stream it ran
    hipEvent_t done = nullptr;
    bool pending = false;
    // evaluations on the library stream since (which lives as long as the process:
    // they need an event only when another stream's evaluation follows)
    bool on_lib = false;
    virtual ~GpuObj() {
        if (done)
            (void)hipEventDestroy(done);
    }
};

// Evaluations of one plan share its scratch, staging and work buffers, so they
// execute on the GPU in the order they were enqueued, whichever stream each
// call names: under the plan's mutex, every evaluation's stream first waits for
// the plan's previous evaluation (an event), and the evaluation records the
// event again once its work is enqueued.  Buffer growth frees the old buffer
// only after the whole device is idle (DevBuf::release).
struct PlanOrder {
    GpuObj* g;
    hipStream_t s;
    bool ok = false, idle = false;
    PlanOrder(GpuObj* obj, hipStream_t st) : g(obj), s(st) {
        if (!g->done && hipEventCreateWithFlags(&g->done, hipEventDisableTiming) != hipSuccess) {
            g->done = nullptr;
            (void)hipGetLastError();
            set_error("plan ordering event: hipEventCreate failed");
            return;
        }
        if (g->on_lib && s != default_stream()) {
            // the previous evaluations ran on the library stream without an event
            ok = hip_ok(hipEventRecord(g->done, default_stream()), "plan ordering record") &&
                 hip_ok(hipStreamWaitEvent(s, g->done, 0), "plan ordering wait");
            g->on_lib = !ok;
            g->pending = g->pending || ok;
            return;
        }
        ok = !g->pending || hip_ok(hipStreamWaitEvent(s, g->done, 0), "plan ordering wait");
        if (ok && s == default_stream())
            g->pending = false; // (the library stream is ordered after it from here on)
    }
    // a blocking evaluation's wait: everything the plan has enqueued so far is done
    // (its stream waited for the evaluations before), so no later call has to wait
    // for it and no event is recorded
    bool sync() {
        idle = hip_ok(hipStreamSynchronize(s), "sync");
        return idle;
    }
    ~PlanOrder() {
        if (idle) {
            g->pending = false;
            g->on_lib = false;
        } else if (ok && s == default_stream())
            g->on_lib = true;
        else if (ok && g->done)
            g->pending = hip_ok(hipEventRecord(g->done, s), "plan ordering record") || g->pending;
    }
    PlanOrder(const PlanOrder&) = delete;
    PlanOrder& operator=(const PlanOrder&) = delete;
};

struct CpxObj : GpuObj {
    std::shared_ptr<Plan1D> p;
    std::shared_ptr<Plan1D> p64; // refinement (float build, KFFT_FLAG_GPU_REFINE): FP64 plan
    DevBuf ref_z, ref_r, ref_x, ref_scr;
};

struct SclrObj : GpuObj {
    uint32_t n = 0;
    std::shared_ptr<Plan1D> p; // length n/2 (even) or n (odd)
    DevBuf st;                 // super twiddles of the plan's direction (even n)
};

static std::mutex g_pool_mu;

static void pool_register(kfft_pool_t* A, GpuObj* o) {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    o->next = (GpuObj*)A->gpu;
    A->gpu = o;
}

static void pool_release_gpu(kfft_pool_t* A) {
    GpuObj* o;
    {
        std::lock_guard<std::mutex> lk(g_pool_mu);
        o = (GpuObj*)A->gpu;
        A->gpu = nullptr;
    }
    while (o) {
        GpuObj* n = o->next;
        delete o;
        o = n;
    }
}

// ================================================================= pool
// Bump allocator with the reference's semantics (kfft_pool.c:13-96): `size`
// usable bytes, allocations fail once they would pass the end, clear zeroes
// the area and rewinds.
extern "C" {

KFFT_API kfft_pool_t* kfft_pool_create(const size_t size) {
    const size_t total = sizeof(kfft_pool_t) + size;
    kfft_pool_t* A = (kfft_pool_t*)calloc(1, total);
    if (!A)
        return nullptr;
    A->allocated = total;
    A->align = 0;
    A->head = A->area;
    A->tail = A->area + size;
    A->cur = A->head;
    A->gpu = nullptr;
    return A;
}

KFFT_API void* kfft_pool_alloc(kfft_pool_t* A, const size_t nmem) {
    if (!A || nmem == 0)
        return nullptr;
    std::lock_guard<std::mutex> lk(g_pool_mu);
    if (A->cur + nmem <= A->tail) {
        void* r = A->cur;
        A->cur += nmem;
        return r;
    }
    return nullptr;
}

KFFT_API size_t kfft_pool_empty(const kfft_pool_t* A) { return A ? (size_t)(A->tail - A->cur) : 0; }

KFFT_API void kfft_pool_zmem(const kfft_pool_t* A, void* ptr, const size_t size) {
    if (A && ptr && size > 0 && (uint8_t*)ptr + size <= A->tail)
        memset(ptr, 0, size);
}

KFFT_API void kfft_pool_clear(kfft_pool_t* A) {
    if (!A)
        return;
    pool_release_gpu(A);
    kfft_pool_zmem(A, A->area, (size_t)(A->tail - A->head));
    A->cur = A->head;
}

KFFT_API void kfft_pool_free(kfft_pool_t* A) {
    if (!A)
        return;
    pool_release_gpu(A);
    free(A);
}

} // extern "C"

// Plan creation protocol of the reference (incs/kfft_algo.h:15-51):
//  lenmem == NULL: allocate in A (cleared first under RENEW) or in a new pool
//  lenmem != NULL: create only when A is given and *lenmem >= need (the plan
//                  object then takes *lenmem bytes); else report need in *lenmem
template <typename T>
static T* plan_prepare(uint32_t flags, size_t need, kfft_pool_t* A, size_t* lenmem) {
    T* plan = nullptr;
    kfft_pool_t* mm = nullptr;
    if (lenmem == nullptr) {
        mm = A ? A : kfft_pool_create(need);
        if (mm) {
            if (A && (flags & KFFT_FLAG_RENEW))
                kfft_pool_clear(mm);
            plan = (T*)kfft_pool_alloc(mm, sizeof(T));
        }
        if (plan == nullptr && A == nullptr)
            kfft_pool_free(mm);
    } else {
        if (A && *lenmem >= need) {
            mm = A;
            if (flags & KFFT_FLAG_RENEW)
                kfft_pool_clear(mm);
            plan = (T*)kfft_pool_alloc(mm, *lenmem);
        }
        if (plan == nullptr)
            *lenmem = need;
    }
    if (plan) {
        memset((void*)plan, 0, sizeof(T));
        plan->object.mmgr = mm;
    }
    return plan;
}

template <typename T>
static void plan_terminate(T* plan, kfft_pool_t* A) {
    if (A == nullptr)
        kfft_pool_free(KFFT_PLAN_MMGR(plan));
}

// ======================================================== pointer handling
static bool is_device_ptr(const void* p) {
    if (!p)
        return false;
    hipPointerAttribute_t at;
    memset(&at, 0, sizeof(at));
    hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged;
}

// Stream of a synchronous entry point: the library stream, ordered after all
// work queued so far on the null stream, so that device buffers a caller (or a
// framework on the null stream) has just produced are complete when read.  (The null
// stream waits for blocking streams, hipStreamCreate's, and its query counts their
// unfinished work; non-blocking streams are the caller's to order, as with the event.)
// A null stream with nothing left to run needs no event pair, whose barrier packets
// on two hardware queues cost a short transform more than its kernel (one blocking
// call of 1024 points FP64: 32 us with the pair and an event recorded after the
// wait, 15.8 without either; the kernel takes 5).
static hipStream_t entry_stream() {
    hipStream_t s = default_stream();
    if (hipStreamQuery(nullptr) == hipSuccess)
        return s;
    (void)hipGetLastError(); // (not ready: no error)
    thread_local hipEvent_t ev = nullptr;
    if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
        ev = nullptr;
        (void)hipStreamSynchronize(nullptr);
        return s;
    }
    if (hipEventRecord(ev, nullptr) != hipSuccess || hipStreamWaitEvent(s, ev, 0) != hipSuccess)
        (void)hipStreamSynchronize(nullptr);
    return s;
}

static kfft_return_t gpu_fail(const char* what) {
    if (what)
        set_error(std::string(what) + ": " + last_error());
    return KFFT_RET_GPU_FAIL;
}

// Maps caller buffers to device buffers for one call, staging host memory.
struct Staged {
    const void* dev = nullptr;
    void* host_out = nullptr;
    size_t bytes = 0;
    bool staged = false;
};

static bool stage_in(const void* user, size_t bytes, DevBuf& buf, Staged& s, hipStream_t st) {
    s.bytes = bytes;
    if (is_device_ptr(user)) {
        s.dev = user;
        return true;
    }
    if (!buf.ensure(bytes))
        return false;
    if (!hip_ok(hipMemcpyAsync(buf.p, user, bytes, hipMemcpyHostToDevice, st), "stage in"))
        return false;
    s.dev = buf.p;
    s.staged = true;
    return true;
}

static bool stage_out(void* user, size_t bytes, DevBuf& buf, Staged& s) {
    s.bytes = bytes;
    if (is_device_ptr(user)) {
        s.dev = user;
        return true;
    }
    if (!buf.ensure(bytes))
        return false;
    s.dev = buf.p;
    s.host_out = user;
    s.staged = true;
    return true;
}

static bool finish_out(const Staged& s, hipStream_t st) {
    if (s.host_out &&
        !hip_ok(hipMemcpyAsync(s.host_out, s.dev, s.bytes, hipMemcpyDeviceToHost, st), "stage out"))
        return false;
    return true;
}

// ======================================================= complex 1D helpers
static size_t cpx_plan_bytes(uint32_t n) { return sizeof(kfft_plan_cpx) + CPXB * n; }

// KFFT_SQRT of the reference's default build (math/kfft_custom_math.h:43-67):
// bisection in kfft_scalar arithmetic (double, or float in the KFFT_HALF_SCALAR
// build) until the bracket is at most 0.001 wide.  Where the float spacing near
// the root exceeds that (x > 2^28) the reference's loop never ends; this one
// stops once the midpoint equals an end of the bracket.
static kfft_scalar bisect_sqrt(kfft_scalar x) {
    if (x <= 0)
        return 0;
    const kfft_scalar acc = (kfft_scalar)0.001;
    kfft_scalar lo = 1, hi = 1;
    if (x < 1)
        lo = x;
    else
        hi = x;
    while ((hi - lo) > acc) {
        const kfft_scalar mid = (lo + hi) / 2;
        if (mid == lo || mid == hi)
            break;
        if (mid * mid > x)
            hi = mid;
        else
            lo = mid;
    }
    return (lo + hi) / 2;
}

// Reference factor list (kfft_cpx.c:103-143) for the public `factors` field,
// with the reference's floor_sqrt (kfft_cpx.c:111: KFFT_SQRT((double)nfft),
// truncated); the engine plans its own radices.
static void fill_factors(kfft_plan_cpx* P) {
    uint32_t p = 4, n = P->nfft;
    const uint32_t lim = (uint32_t)bisect_sqrt((kfft_scalar)(double)P->nfft);
    P->fac_count = 0;
    P->prm_count = 0;
    if (n == 0)
        return;
    do {
        while (n % p) {
            if (p == 4)
                p = 2;
            else if (p == 2)
                p = 3;
            else
                p += 2;
            if (p > lim)
                p = n;
        }
        if (P->level < KFFT_PLAN_LEVEL && p > KFFT_BFLY_LEVEL && p >= KFFT_RADER_LIMIT &&
            P->prm_count < MAX_ROOTS)
            P->primes[P->prm_count++].prime = p;
        n /= p;
        if (P->fac_count < MAX_FACTORS) {
            P->factors[2 * P->fac_count] = p;
            P->factors[2 * P->fac_count + 1] = n;
            P->fac_count++;
        }
    } while (n > 1);
}

static void host_twiddles(kfft_cpx* tw, uint32_t n, bool inverse) {
    const long double two_pi = 6.283185307179586476925286766559005768L;
    auto fill = [=](uint32_t i0, uint32_t i1) {
        for (uint32_t i = i0; i < i1; ++i) {
            long double a = two_pi * (long double)i / (long double)n;
            tw[i].r = (kfft_scalar)cosl(a);
            tw[i].i = (kfft_scalar)(inverse ? sinl(a) : -sinl(a));
        }
    };
    // large tables (plans beyond a few million points) in parallel slices; every
    // entry is computed the same way either way
    const uint32_t hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    if (n < (1u << 20) || hw == 1) {
        fill(0, n);
        return;
    }
    std::vector<std::thread> th;
    const uint32_t step = (n + hw - 1) / hw;
    for (uint32_t t = 0; t < hw; ++t) {
        const uint32_t i0 = t * step, i1 = std::min(n, i0 + step);
        if (i0 < i1)
            th.emplace_back(fill, i0, i1);
    }
    for (auto& x : th)
        x.join();
}

// radix-16 arithmetic of the precision form (float build only; the double
// build's data is FP64 and always runs the FP64 passes)
static uint32_t split_dft(uint32_t flags) {
    if (PREC != 4)
        return 0;
    if (flags & KFFT_FLAG_GPU_SPLIT_F16)
        return KFA_FAST_MFMA_F16;
    if (flags & KFFT_FLAG_GPU_SPLIT_BF16)
        return KFA_FAST_MFMA_BF16;
    return 0;
}

// The entry points of plans created with a split-operand flag run the radix-16
// stages of every transform they make (rows, columns, real, convolution) as
// split matrix products (float build; the double build ignores the flags).
struct SplitScope {
    explicit SplitScope(uint32_t flags) { set_split_dft(split_dft(flags)); }
    ~SplitScope() { set_split_dft(0); }
    SplitScope(const SplitScope&) = delete;
    SplitScope& operator=(const SplitScope&) = delete;
};

static double cpx_scale(const kfft_plan_cpx* P) {
    if ((P->flags & KFFT_FLAG_INVERSE) && !(P->flags & KFFT_FLAG_DISABLE_NORM))
        return 1.0 / (double)P->nfft;
    return 1.0;
}

static Layout contiguous(const void* p, int64_t dist, uint32_t flags = 0) {
    Layout l;
    l.ptr = (void*)p;
    l.dist_hi = dist;
    l.dist_lo = 0;
    l.stride = 1;
    l.C = 1;
    l.flags = flags;
    return l;
}

// [p, p + np) and [q, q + nq) have bytes in common
static bool overlap(const void* p, size_t np, const void* q, size_t nq) {
    return (const char*)p < (const char*)q + nq && (const char*)q < (const char*)p + np;
}

// Scratch for `batch` rows of a plan in buf, past its first `off` bytes: how many rows
// may run at a time, 0 without room.  Bluestein on a power-of-two convolution length
// takes up to twice the shortest length's scratch; where that does not fit, groups of
// the batch run in what the shortest length would take.
static uint64_t scratch_group(const Plan1D& pl, DevBuf& buf, size_t off, uint64_t batch) {
    if (buf.ensure(off + pl.scratch_bytes(batch)))
        return batch;
    const uint64_t g = pl.group_within(batch, pl.scratch_charge(batch));
    return g < batch && buf.ensure(off + pl.scratch_bytes(g)) ? g : 0;
}

// The rows of a batch, `group` at a time in the same scratch.  Groups whose output
// lies over other groups' input run from the end that is not read again; that end
// exists where both sides' rows are equally far apart.
static hipError_t run_groups(const Plan1D& pl, const Layout& in, const Layout& out, uint64_t batch,
                             uint64_t group, bool inverse, double scale, void* scratch,
                             hipStream_t s, const Fuse* fz = nullptr) {
    if (group >= batch)
        return pl.execute(in, out, batch, inverse, scale, scratch, s, fz);
    const int64_t eb = 2 * pl.prec();
    const int64_t id = in.dist_hi * ((in.flags & KFA_IO_REAL) ? eb / 2 : eb);
    const int64_t od = out.dist_hi * ((out.flags & KFA_IO_REAL) ? eb / 2 : eb);
    if (id != od && overlap(in.ptr, (size_t)batch * id, out.ptr, (size_t)batch * od))
        return hipErrorOutOfMemory;
    const uint64_t n = (batch + group - 1) / group;
    const bool up = out.ptr > in.ptr;
    for (uint64_t k = 0; k < n; ++k) {
        const uint64_t b0 = (up ? n - 1 - k : k) * group;
        Layout i = in, o = out;
        i.ptr = (char*)in.ptr + (int64_t)b0 * id;
        o.ptr = (char*)out.ptr + (int64_t)b0 * od;
        const hipError_t e = pl.execute(i, o, std::min(group, batch - b0), inverse, scale, scratch,
                                        s, fz);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

// The precision form with one refinement step (float build): y0 = T(x) in
// FP32, the residual r = x - T^-1(y0) with T^-1 evaluated in FP64, then
// y = y0 + T(r).  T^-1 of a forward plan is the inverse scaled by 1/N; of a
// normalised inverse, the forward; of an unnormalised inverse, the forward
// scaled by 1/N.  Runs in chunks of about 256 MiB of FP32 data.
static kfft_return_t cpx_refine(kfft_plan_cpx* P, CpxObj* g, const void* din, void* dout,
                                uint32_t batch, hipStream_t s, const Fuse& fz) {
    const uint32_t n = P->nfft;
    const bool inverse = (P->flags & KFFT_FLAG_INVERSE) != 0;
    const double inv_scale =
        (!inverse || (P->flags & KFFT_FLAG_DISABLE_NORM)) ? 1.0 / (double)n : 1.0;
    const size_t inst32 = (size_t)n * 8, inst64 = (size_t)n * 16;
    const uint32_t chunk =
        (uint32_t)std::max<size_t>(1, std::min<size_t>(batch, ((size_t)256 << 20) / inst32));
    const bool alias = din == dout;
    if (!g->scratch.ensure(std::max(g->p->scratch_bytes(chunk), g->p64->scratch_bytes(chunk))) ||
        !g->ref_z.ensure(inst64 * chunk) || !g->ref_r.ensure(inst32 * chunk) ||
        (alias && !g->ref_x.ensure(inst32 * chunk)))
        return gpu_fail("refinement buffers");
    for (uint32_t c0 = 0; c0 < batch; c0 += chunk) {
        const uint32_t nb = std::min(chunk, batch - c0);
        const uint64_t cnt = (uint64_t)n * nb;
        const char* x = (const char*)din + (size_t)c0 * inst32;
        char* y = (char*)dout + (size_t)c0 * inst32;
        if (alias) {
            if (!hip_ok(launch_copy(4, x, g->ref_x.p, cnt, 0, 1.0, s), "refine save"))
                return KFFT_RET_GPU_FAIL;
            x = (const char*)g->ref_x.p;
        }
        if (!hip_ok(g->p->execute(contiguous(x, n), contiguous(y, n), nb, inverse, cpx_scale(P),
                                  g->scratch.p, s, &fz), "refine y0") ||
            !hip_ok(launch_widen(y, g->ref_z.p, cnt, s), "refine widen") ||
            !hip_ok(g->p64->execute(contiguous(g->ref_z.p, n), contiguous(g->ref_z.p, n), nb,
                                    !inverse, inv_scale, g->scratch.p, s), "refine residual fft") ||
            !hip_ok(launch_residual(x, g->ref_z.p, g->ref_r.p, cnt, s), "refine residual") ||
            !hip_ok(g->p->execute(contiguous(g->ref_r.p, n), contiguous(g->ref_r.p, n), nb, inverse,
                                  cpx_scale(P), g->scratch.p, s, &fz), "refine correction") ||
            !hip_ok(launch_accumulate(y, g->ref_r.p, cnt, s), "refine add"))
            return KFFT_RET_GPU_FAIL;
    }
    return KFFT_RET_SUCCESS;
}

// Batched complex transform on device pointers, on stream s, no sync.
static kfft_return_t cpx_run_dev(kfft_plan_cpx* P, const void* din, void* dout, uint32_t batch,
                                 hipStream_t s) {
    CpxObj* g = (CpxObj*)P->gpu;
    if (!g || !g->p)
        return KFFT_RET_BADARGUMENTS;
    const Plan1D& pl = *g->p;
    Fuse fz;
    fz.onchip = (P->flags & KFFT_FLAG_GPU_ONCHIP) != 0;
    fz.dft = split_dft(P->flags);
    const bool inverse = (P->flags & KFFT_FLAG_INVERSE) != 0;
    if (g->p64)
        return cpx_refine(P, g, din, dout, batch, s, fz);
    const uint64_t group = scratch_group(pl, g->scratch, 0, batch);
    if (!group && batch)
        return gpu_fail("scratch");
    hipError_t e = run_groups(pl, contiguous(din, P->nfft), contiguous(dout, P->nfft), batch, group,
                              inverse, cpx_scale(P), g->scratch.p, s, &fz);
    return hip_ok(e, "cpx execute") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

static kfft_return_t cpx_run(kfft_plan_cpx* P, const kfft_cpx* fin, kfft_cpx* fout,
                             uint32_t batch) {
    if (!P || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    CpxObj* g = (CpxObj*)P->gpu;
    if (!g)
        return KFFT_RET_BADARGUMENTS;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(P->flags);
    const size_t bytes = (size_t)P->nfft * CPXB * batch;
    Staged si, so;
    if (!stage_in(fin, bytes, g->stage_in, si, s) || !stage_out(fout, bytes, g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = cpx_run_dev(P, si.dev, (void*)so.dev, batch, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    if (!finish_out(so, s) || !order.sync())
        return KFFT_RET_GPU_FAIL;
    if (g->p->async_error()) {
        set_error("fused transform: a dependency wait timed out");
        return KFFT_RET_GPU_FAIL;
    }
    return KFFT_RET_SUCCESS;
}

// The plan of an ordinary transform; a Bluestein length whose power-of-two convolution
// finds no room for its tables and one transform takes the shortest one.
static std::shared_ptr<Plan1D> default_plan(uint32_t n, int prec) {
    const PlanVariant v = default_variant(n, prec);
    std::shared_ptr<Plan1D> p = get_plan(n, prec, v);
    if (!v.pow2_m || (p && p->scratch_bytes(1) <= device_room()))
        return p;
    p.reset();
    return get_plan(n, prec);
}

static kfft_plan_cpx* config_cpx(uint32_t nfft, uint32_t flags, kfft_pool_t* A, size_t* lenmem) {
    const size_t need = cpx_plan_bytes(nfft);
    kfft_plan_cpx* P = plan_prepare<kfft_plan_cpx>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = nfft;
    P->flags = flags;
    P->level = 0;
    fill_factors(P);
    P->twiddles = (kfft_cpx*)kfft_pool_alloc(mm, CPXB * nfft);
    if (!P->twiddles) {
        plan_terminate(P, A);
        return nullptr;
    }
    host_twiddles(P->twiddles, nfft, (flags & KFFT_FLAG_INVERSE) != 0);
    CpxObj* g = new (std::nothrow) CpxObj();
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    PlanVariant split;
    split.maxr = KFA_MAXR_SPLIT; // as many radix-16 stages as the length allows
    g->p = split_dft(flags) ? get_plan(nfft, PREC, split) : default_plan(nfft, PREC);
    if (PREC == 4 && (flags & KFFT_FLAG_GPU_REFINE))
        g->p64 = default_plan(nfft, 8);
    if (!g->p || (PREC == 4 && (flags & KFFT_FLAG_GPU_REFINE) && !g->p64)) {
        delete g;
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

// ======================================================= scalar 1D helpers
static size_t sclr_plan_bytes(uint32_t n) {
    if (n % 2)
        return sizeof(kfft_plan_sclr) + cpx_plan_bytes(n);
    return sizeof(kfft_plan_sclr) + cpx_plan_bytes(n / 2) + CPXB * (n / 2);
}

static uint32_t sclr_out_len(const kfft_plan_sclr* P) {
    if ((P->nfft % 2) || (P->flags & KFFT_FLAG_EXPAND_SCALAR))
        return P->nfft;
    return P->nfft / 2 + 1;
}

static double sclr_scale(const kfft_plan_sclr* P) {
    if (P->flags & KFFT_FLAG_DISABLE_NORM)
        return 1.0;
    return 1.0 / (double)((P->nfft % 2) ? P->nfft : P->nfft / 2);
}

// Forward real transform of `batch` rows (input distance n reals) into
// complex rows of distance out_dist.  expand: full-spectrum mirror.  blk4 (plans
// with sclr_fuses_blocked): the rows as columns in blocks of four (KFA_IO_BLK4).
static bool sclr_fuses_blocked(const kfft_plan_sclr* P) {
    return P->nfft % 2 == 0 && ((SclrObj*)P->gpu)->p->fuses_real_post();
}
// Real and complex rows of one batch lie at different distances.  Where the output
// lies over the input (over), a pass's stores would reach rows that another
// workgroup or group has still to read, so the transforms (odd lengths of the
// inverse: their input) go through scratch; without room for that, the passes run as
// they do on buffers apart, each reading its own rows before it stores them.
static kfft_return_t sclr_fwd_dev(kfft_plan_sclr* P, const void* din, void* dout, uint32_t batch,
                                  int64_t out_dist, bool expand, hipStream_t s,
                                  bool blk4 = false) {
    SclrObj* g = (SclrObj*)P->gpu;
    const Plan1D& pl = *g->p;
    const uint32_t n = P->nfft, h = n / 2;
    const uint32_t ol = (n % 2 || expand) ? n : h + 1;
    const bool over = batch > 1 && !blk4 &&
                      overlap(din, (size_t)batch * n * sizeof(kfft_scalar), dout,
                              ((size_t)(batch - 1) * out_dist + ol) * CPXB);
    // (the two-pass form with the rebuild reads a whole batch before it stores any)
    if (over && (expand || !pl.fuses_real_post_shaped())) {
        const uint32_t zl = n % 2 ? n : h;
        const size_t zbytes = ((size_t)batch * zl * CPXB + 255) / 256 * 256;
        if (g->scratch.ensure(zbytes + pl.scratch_bytes(batch))) {
            void* z = g->scratch.p;
            hipError_t e = pl.execute(contiguous(din, zl, n % 2 ? KFA_IO_REAL : 0),
                                      contiguous(z, zl), batch, false, 1.0,
                                      (char*)g->scratch.p + zbytes, s);
            if (e == hipSuccess && n % 2 == 0)
                e = launch_real_post(PREC, z, h, dout, out_dist, 0, 1, 1, h, batch, g->st.p,
                                     expand ? 1 : 0, 0, s);
            else if (e == hipSuccess) // (rows of n, as both callers have them)
                e = launch_copy(PREC, z, dout, (uint64_t)batch * n, 0, 1.0, s);
            return hip_ok(e, "scalar fwd") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
        }
    }
    const uint64_t group = scratch_group(pl, g->scratch, 0, batch);
    if (!group && batch)
        return gpu_fail("scratch");
    if (n % 2) {
        hipError_t e = run_groups(pl, contiguous(din, n, KFA_IO_REAL), contiguous(dout, out_dist),
                                  batch, group, false, 1.0, g->scratch.p, s);
        return hip_ok(e, "scalar fwd") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    // (compiled lengths: one pass with the rebuild in its store against the shaped row
    // pass and a rebuild sweep, forward and inverse 4096 x 4096 FP32 108 us, 77 with
    // both rebuilds in the passes; 128 x 131072 FP64 240 and 132)
    if (!expand && ((pl.fuses_real_post() &&
                     (blk4 || !pl.shaped_rows() || (pl.fuses_real_pre() && !over))) ||
                    pl.fuses_real_post_shaped())) {
        // one LDS pass, or the shaped two-pass form: Z = FFT_h(x viewed as h complex)
        // rebuilt into X in the last pass's store
        Layout o = contiguous(dout, out_dist);
        o.real_post = g->st.p;
        if (blk4) {
            o.dist_hi = 4;
            o.stride = 4 * (int64_t)batch;
            o.flags |= KFA_IO_BLK4;
        }
        hipError_t e = pl.execute(contiguous(din, h), o, batch, false, 1.0, g->scratch.p, s);
        return hip_ok(e, "scalar fwd") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    // Z = FFT_h(x viewed as h complex), written where X goes, then rebuilt in place
    hipError_t e = run_groups(pl, contiguous(din, h), contiguous(dout, out_dist), batch, group,
                              false, 1.0, g->scratch.p, s);
    if (!hip_ok(e, "scalar fwd fft"))
        return KFFT_RET_GPU_FAIL;
    e = launch_real_post(PREC, dout, out_dist, dout, out_dist, 0, 1, 1, h, batch, g->st.p,
                         expand ? 1 : 0, 0, s);
    return hip_ok(e, "scalar post") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

// Inverse real transform: complex rows (distance in_dist, first n/2+1 used
// for even n) to real rows of n.  pw: null, or a spectrum in din's layout
// that multiplies din on the way in (a convolution's product); it is applied
// in the first kernel that reads din where the plan allows, else by a
// separate sweep into din (with pw given, din is the caller's work buffer).
static void hadamard_dev(void* acc, const void* other, uint64_t n, hipStream_t s);
static kfft_return_t sclr_inv_dev(kfft_plan_sclr* P, const void* din, int64_t in_dist, void* dout,
                                  uint32_t batch, hipStream_t s, const void* pw = nullptr,
                                  bool blk4 = false) {
    SclrObj* g = (SclrObj*)P->gpu;
    const Plan1D& pl = *g->p;
    const uint32_t n = P->nfft;
    const double sc = sclr_scale(P);
    if (n % 2) {
        if (batch > 1 && !pw &&
            overlap(din, ((size_t)(batch - 1) * in_dist + n) * CPXB, dout,
                    (size_t)batch * n * sizeof(kfft_scalar))) {
            const size_t xbytes = ((size_t)batch * in_dist * CPXB + 255) / 256 * 256;
            if (g->scratch.ensure(xbytes + pl.scratch_bytes(batch))) {
                void* x = g->scratch.p;
                hipError_t e = launch_copy(PREC, din, x, (uint64_t)(batch - 1) * in_dist + n, 0,
                                           1.0, s);
                if (e == hipSuccess)
                    e = pl.execute(contiguous(x, in_dist), contiguous(dout, n, KFA_IO_REAL), batch,
                                   true, sc, (char*)g->scratch.p + xbytes, s);
                return hip_ok(e, "scalar inv") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
            }
        }
        const uint64_t group = scratch_group(pl, g->scratch, 0, batch);
        if (!group && batch)
            return gpu_fail("scratch");
        Fuse fz;
        if (pw && (pl.kind() == Kind::Direct || pl.kind() == Kind::Identity))
            fz.pw_in = pw;
        else if (pw)
            hadamard_dev(const_cast<void*>(din), pw, (uint64_t)in_dist * batch, s);
        hipError_t e = run_groups(pl, contiguous(din, in_dist), contiguous(dout, n, KFA_IO_REAL),
                                  batch, group, true, sc, g->scratch.p, s, &fz);
        return hip_ok(e, "scalar inv") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    const uint32_t h = n / 2;
    // the inverse rebuild in the pass's load (one read of the spectrum, one write of
    // the signal, against a sweep through a work buffer before the pass), unless the
    // output lies over spectra still to be read
    if (!pw && pl.fuses_real_pre() &&
        !overlap(din, (size_t)batch * (blk4 ? (h + 4) / 4 * 4 : in_dist) * CPXB, dout,
                 (size_t)batch * n * sizeof(kfft_scalar))) {
        if (!g->scratch.ensure(pl.scratch_bytes(batch)))
            return gpu_fail("scratch");
        Layout in = contiguous(din, blk4 ? 4 : in_dist);
        in.real_pre = g->st.p;
        if (blk4) {
            in.stride = 4 * (int64_t)batch;
            in.flags |= KFA_IO_BLK4;
        }
        hipError_t e = pl.execute(in, contiguous(dout, h), batch, true, sc, g->scratch.p, s);
        return hip_ok(e, "scalar inv") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    const size_t zbytes = ((size_t)batch * h * CPXB + 255) / 256 * 256;
    const uint64_t group = scratch_group(pl, g->scratch, zbytes, batch);
    if (!group && batch)
        return gpu_fail("scratch");
    void* z = g->scratch.p;
    void* scr = (char*)g->scratch.p + zbytes;
    hipError_t e = launch_real_pre(PREC, din, blk4 ? 4 : in_dist, 0, blk4 ? 4 * (int64_t)batch : 1,
                                   1, z, h, h, batch, g->st.p, pw, s, blk4 ? 1 : 0);
    if (!hip_ok(e, "scalar pre"))
        return KFFT_RET_GPU_FAIL;
    e = run_groups(pl, contiguous(z, h), contiguous(dout, h), batch, group, true, sc, scr, s);
    return hip_ok(e, "scalar inv fft") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

static kfft_plan_sclr* config_sclr(uint32_t nfft, uint32_t flags, kfft_pool_t* A, size_t* lenmem) {
    const size_t need = sclr_plan_bytes(nfft);
    kfft_plan_sclr* P = plan_prepare<kfft_plan_sclr>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = nfft;
    P->flags = flags;
    const uint32_t blen = (nfft % 2) ? nfft : nfft / 2;
    P->basis = config_cpx(blen, KFFT_CHECK_FLAGS(flags), mm, nullptr);
    if (!P->basis) {
        plan_terminate(P, A);
        return nullptr;
    }
    SclrObj* g = new (std::nothrow) SclrObj();
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    g->n = nfft;
    g->p = ((CpxObj*)P->basis->gpu)->p;
    if (nfft % 2 == 0) {
        const uint32_t h = nfft / 2;
        P->super_twiddles = (kfft_cpx*)kfft_pool_alloc(mm, CPXB * h);
        if (!P->super_twiddles || !make_real_twiddles(g->st, h, PREC, (flags & KFFT_FLAG_INVERSE) != 0)) {
            delete g;
            plan_terminate(P, A);
            return nullptr;
        }
        const long double pi = 3.141592653589793238462643383279502884L;
        for (uint32_t i = 0; i < h; ++i) {
            long double ph = -pi * ((long double)(i + 1) / h + 0.5L);
            if (flags & KFFT_FLAG_INVERSE)
                ph = -ph;
            P->super_twiddles[i].r = (kfft_scalar)cosl(ph);
            P->super_twiddles[i].i = (kfft_scalar)sinl(ph);
        }
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

static kfft_return_t sclr_fwd(kfft_plan_sclr* P, const kfft_scalar* fin, kfft_cpx* fout,
                              uint32_t batch) {
    if (!P || !fin || !fout || !P->gpu)
        return KFFT_RET_BADARGUMENTS;
    if (P->basis->flags & KFFT_FLAG_INVERSE)
        return KFFT_RET_IMPROPER_PLAN;
    SclrObj* g = (SclrObj*)P->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(P->flags);
    const uint32_t ol = sclr_out_len(P);
    Staged si, so;
    if (!stage_in(fin, (size_t)P->nfft * sizeof(kfft_scalar) * batch, g->stage_in, si, s) ||
        !stage_out(fout, (size_t)ol * CPXB * batch, g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = sclr_fwd_dev(P, si.dev, (void*)so.dev, batch, ol,
                                   (P->flags & KFFT_FLAG_EXPAND_SCALAR) != 0, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    if (!finish_out(so, s) || !order.sync())
        return KFFT_RET_GPU_FAIL;
    return KFFT_RET_SUCCESS;
}

static kfft_return_t sclr_inv(kfft_plan_sclr* P, const kfft_cpx* fin, kfft_scalar* fout,
                              uint32_t batch) {
    if (!P || !fin || !fout || !P->gpu)
        return KFFT_RET_BADARGUMENTS;
    if (!(P->basis->flags & KFFT_FLAG_INVERSE))
        return KFFT_RET_IMPROPER_PLAN;
    SclrObj* g = (SclrObj*)P->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(P->flags);
    const uint32_t il = sclr_out_len(P);
    Staged si, so;
    if (!stage_in(fin, (size_t)il * CPXB * batch, g->stage_in, si, s) ||
        !stage_out(fout, (size_t)P->nfft * sizeof(kfft_scalar) * batch, g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = sclr_inv_dev(P, si.dev, il, (void*)so.dev, batch, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    if (!finish_out(so, s) || !order.sync())
        return KFFT_RET_GPU_FAIL;
    return KFFT_RET_SUCCESS;
}

// ============================================================== 2D helpers
// Column transforms of a y-by-x row-major complex matrix (batch `nmat`),
// in place: strided LDS passes when the column plan allows it, otherwise
// transpose / rows / transpose through `work`.
// Columns longer than the shaped one-pass lengths run as a column four-step
// (two passes whose lanes walk the columns) rather than the one-pass kernel,
// whose workgroups would each walk a single column.
static const Plan1D& column_plan(const Plan1D& py) {
    if (py.kind() != Kind::Direct || py.two_pass() || py.n() <= 4096)
        return py;
    static std::mutex mu;
    static std::map<std::pair<uint32_t, int>, std::shared_ptr<Plan1D>> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_pair(py.n(), py.prec());
    auto it = cache.find(key);
    if (it == cache.end()) {
        PlanVariant v;
        v.four = true;
        std::shared_ptr<Plan1D> p = get_plan(py.n(), py.prec(), v);
        it = cache.emplace(key, (p && p->supports_plain_columns()) ? p : nullptr).first;
    }
    return it->second ? *it->second : py;
}

static kfft_return_t cols_cpx_dev(const Plan1D& py_, void* data, uint32_t x, uint32_t y,
                                  uint32_t nmat, bool inverse, double scale, DevBuf& scratch,
                                  DevBuf& work, hipStream_t s) {
    const Plan1D& py = column_plan(py_);
    if (py.supports_plain_columns()) {
        if (!scratch.ensure(py.scratch_bytes((uint64_t)x * nmat)))
            return gpu_fail("scratch");
        Layout l;
        l.ptr = data;
        l.C = x;
        l.dist_hi = (int64_t)x * y;
        l.dist_lo = 1;
        l.stride = x;
        hipError_t e = py.execute(l, l, (uint64_t)x * nmat, inverse, scale, scratch.p, s);
        return hip_ok(e, "columns") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    const size_t bytes = (size_t)x * y * nmat * CPXB;
    const uint64_t cols = (uint64_t)x * nmat;
    const uint64_t group = work.ensure(bytes) ? scratch_group(py, scratch, 0, cols) : 0;
    if (!group && cols)
        return gpu_fail("work");
    if (!hip_ok(launch_transpose((int)CPXB, data, work.p, x, y, nmat, s), "transpose"))
        return KFFT_RET_GPU_FAIL;
    hipError_t e = run_groups(py, contiguous(work.p, y), contiguous(work.p, y), cols, group,
                              inverse, scale, scratch.p, s);
    if (!hip_ok(e, "transposed columns"))
        return KFFT_RET_GPU_FAIL;
    return hip_ok(launch_transpose((int)CPXB, work.p, data, y, x, nmat, s), "transpose back")
               ? KFFT_RET_SUCCESS
               : KFFT_RET_GPU_FAIL;
}

struct C2dObj : GpuObj {};

static size_t c2d_plan_bytes(uint32_t x, uint32_t y) {
    size_t r = sizeof(kfft_plan_c2d) + cpx_plan_bytes(x);
    if (x != y)
        r += cpx_plan_bytes(y);
    return r;
}

// Row plans that can multiply their input by a second spectrum as they load it
// (Fuse::pw_in): one- and two-pass transforms.
static bool rows_take_product(const Plan1D& p) {
    return p.kind() == Kind::Direct || p.kind() == Kind::Identity;
}

// pw: null, or a spectrum in din's layout multiplied in by the row pass's load
// (only where rows_take_product holds for the row plan)
static kfft_return_t c2d_run_dev(kfft_plan_c2d* P, const void* din, void* dout, hipStream_t s,
                                 const void* pw = nullptr) {
    C2dObj* g = (C2dObj*)P->gpu;
    const Plan1D& px = *((CpxObj*)P->plan_x->gpu)->p;
    const Plan1D& py = *((CpxObj*)P->plan_y->gpu)->p;
    const bool inv = (P->flags & KFFT_FLAG_INVERSE) != 0;
    const bool norm = inv && !(P->flags & KFFT_FLAG_DISABLE_NORM);
    const uint64_t group = scratch_group(px, g->scratch, 0, P->y);
    if (!group)
        return gpu_fail("scratch");
    Fuse fz;
    fz.pw_in = pw;
    hipError_t e = run_groups(px, contiguous(din, P->x), contiguous(dout, P->x), P->y, group, inv,
                              norm ? 1.0 / P->x : 1.0, g->scratch.p, s, &fz);
    if (!hip_ok(e, "2d rows"))
        return KFFT_RET_GPU_FAIL;
    return cols_cpx_dev(py, dout, P->x, P->y, 1, inv, norm ? 1.0 / P->y : 1.0, g->scratch,
                        g->work_a, s);
}

static kfft_plan_c2d* config2_cpx(uint32_t x, uint32_t y, uint32_t flags, kfft_pool_t* A,
                                  size_t* lenmem) {
    kfft_plan_c2d* P = plan_prepare<kfft_plan_c2d>(flags, c2d_plan_bytes(x, y), A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = x * y;
    P->x = x;
    P->y = y;
    P->flags = flags;
    P->plan_x = config_cpx(x, KFFT_CHECK_FLAGS(flags), mm, nullptr);
    P->plan_y = (x == y) ? P->plan_x : config_cpx(y, KFFT_CHECK_FLAGS(flags), mm, nullptr);
    C2dObj* g = (P->plan_x && P->plan_y) ? new (std::nothrow) C2dObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

static kfft_return_t c2d_run(kfft_plan_c2d* P, const kfft_cpx* fin, kfft_cpx* fout) {
    if (!P || !fin || !fout || !P->gpu)
        return KFFT_RET_BADARGUMENTS;
    C2dObj* g = (C2dObj*)P->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(P->flags);
    const size_t bytes = (size_t)P->nfft * CPXB;
    Staged si, so;
    if (!stage_in(fin, bytes, g->stage_in, si, s) || !stage_out(fout, bytes, g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = c2d_run_dev(P, si.dev, (void*)so.dev, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    if (!finish_out(so, s) || !order.sync())
        return KFFT_RET_GPU_FAIL;
    return KFFT_RET_SUCCESS;
}

// --- 2D real ---------------------------------------------------------------
struct S2dObj : GpuObj {};

static size_t s2d_plan_bytes(uint32_t x, uint32_t y, uint32_t flags) {
    if (flags & KFFT_FLAG_INVERSE)
        return sizeof(kfft_plan_s2d) + cpx_plan_bytes(x) + sclr_plan_bytes(y);
    return sizeof(kfft_plan_s2d) + sclr_plan_bytes(x) + cpx_plan_bytes(y);
}

static kfft_plan_s2d* config2_sclr(uint32_t x, uint32_t y, uint32_t flags, kfft_pool_t* A,
                                   size_t* lenmem) {
    kfft_plan_s2d* P = plan_prepare<kfft_plan_s2d>(flags, s2d_plan_bytes(x, y, flags), A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = x * y;
    P->x = x;
    P->y = y;
    P->flags = flags;
    const uint32_t f = KFFT_CHECK_FLAGS(flags);
    if (flags & KFFT_FLAG_INVERSE) {
        P->plan_x = (kfft_object_t*)config_cpx(x, f, mm, nullptr);
        P->plan_y = (kfft_object_t*)config_sclr(y, f | KFFT_FLAG_EXPAND_SCALAR, mm, nullptr);
    } else {
        P->plan_x = (kfft_object_t*)config_sclr(x, f | KFFT_FLAG_EXPAND_SCALAR, mm, nullptr);
        P->plan_y = (kfft_object_t*)config_cpx(y, f, mm, nullptr);
    }
    S2dObj* g = (P->plan_x && P->plan_y) ? new (std::nothrow) S2dObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

// forward: real rows with full-spectrum rows, then complex columns
static kfft_return_t s2d_fwd_dev(kfft_plan_s2d* P, const void* din, void* dout, hipStream_t s) {
    S2dObj* g = (S2dObj*)P->gpu;
    kfft_plan_sclr* sx = (kfft_plan_sclr*)P->plan_x;
    kfft_plan_cpx* cy = (kfft_plan_cpx*)P->plan_y;
    kfft_return_t r = sclr_fwd_dev(sx, din, dout, P->y, P->x, true, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return cols_cpx_dev(*((CpxObj*)cy->gpu)->p, dout, P->x, P->y, 1, false, 1.0, g->scratch,
                        g->work_a, s);
}

// inverse: complex rows, then real columns (rebuilt half spectrum per column)
static kfft_return_t s2d_inv_dev(kfft_plan_s2d* P, const void* din, void* dout, hipStream_t s) {
    S2dObj* g = (S2dObj*)P->gpu;
    kfft_plan_cpx* cx_ = (kfft_plan_cpx*)P->plan_x;
    kfft_plan_sclr* sy = (kfft_plan_sclr*)P->plan_y;
    const Plan1D& px = *((CpxObj*)cx_->gpu)->p;
    SclrObj* gy = (SclrObj*)sy->gpu;
    const Plan1D& py = *gy->p;
    const uint32_t x = P->x, y = P->y;
    const size_t nb = (size_t)x * y * CPXB;
    const uint64_t group = g->work_a.ensure(nb) ? scratch_group(px, g->scratch, 0, y) : 0;
    if (!group)
        return gpu_fail("work");
    hipError_t e = run_groups(px, contiguous(din, x), contiguous(g->work_a.p, x), y, group, true,
                              cpx_scale(cx_), g->scratch.p, s);
    if (!hip_ok(e, "2d inverse rows"))
        return KFFT_RET_GPU_FAIL;
    const double sc = sclr_scale(sy);
    if (!py.supports_columns()) {
        // transpose to column-major rows, real inverse rows, real transpose back
        if (!g->work_b.ensure(nb))
            return gpu_fail("work");
        if (!hip_ok(launch_transpose((int)CPXB, g->work_a.p, g->work_b.p, x, y, 1, s), "T"))
            return KFFT_RET_GPU_FAIL;
        kfft_return_t r = sclr_inv_dev(sy, g->work_b.p, y, g->work_a.p, x, s);
        if (r != KFFT_RET_SUCCESS)
            return r;
        return hip_ok(launch_transpose((int)sizeof(kfft_scalar), g->work_a.p, dout, y, x, 1, s),
                      "T back")
                   ? KFFT_RET_SUCCESS
                   : KFFT_RET_GPU_FAIL;
    }
    if (y % 2) {
        if (!g->scratch.ensure(py.scratch_bytes(x)))
            return gpu_fail("scratch");
        Layout li, lo;
        li.ptr = g->work_a.p;
        li.C = x;
        li.dist_hi = (int64_t)x * y;
        li.dist_lo = 1;
        li.stride = x;
        lo = li;
        lo.ptr = dout;
        lo.flags = KFA_IO_REAL;
        e = py.execute(li, lo, x, true, sc, g->scratch.p, s);
        return hip_ok(e, "2d inverse columns") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
    }
    const uint32_t h = y / 2;
    const size_t zb = ((size_t)x * h * CPXB + 255) / 256 * 256;
    if (!g->scratch.ensure(zb + py.scratch_bytes(x)))
        return gpu_fail("scratch");
    void* z = g->scratch.p;
    e = launch_real_pre(PREC, g->work_a.p, (int64_t)x * y, 1, x, x, z, h, h, x, gy->st.p, nullptr,
                        s);
    if (!hip_ok(e, "2d column pre"))
        return KFFT_RET_GPU_FAIL;
    Layout lo;
    lo.ptr = dout;
    lo.C = x;
    lo.dist_hi = (int64_t)x * y;
    lo.dist_lo = 1;
    lo.stride = x;
    lo.flags = KFA_IO_REAL_PAIRS;
    e = py.execute(contiguous(z, h), lo, x, true, sc, (char*)g->scratch.p + zb, s);
    return hip_ok(e, "2d inverse columns") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

// ======================================================== convolution
struct ConvObj : GpuObj {
    // real conv2d of even width x: an inverse real plan of length x for the
    // half-spectrum form (own pool, so the caller's plan memory is unchanged)
    kfft_plan_sclr* rows_inv = nullptr;
    DevBuf work_c;   // transposed-column fallback of the half-spectrum form
    ColumnConv cols; // one-pass columns of the half-spectrum form (y == 0: none)
    ~ConvObj() override {
        if (rows_inv)
            kfft_pool_free(KFFT_PLAN_MMGR(rows_inv));
    }
};

static void hadamard_dev(void* acc, const void* other, uint64_t n, hipStream_t s) {
    (void)hip_ok(launch_hadamard(PREC, acc, other, n, s), "hadamard");
}

// ------------------------------------------------------------------ shift
// fftshift / ifftshift of one row (kfft_shift.c:4-61): for even sizes the
// halves swap; for odd sizes the rotation is by floor(n/2) (forward) or
// ceil(n/2) (inverse).  Host buffers.
template <typename T>
static void shift_host(T* buf, uint32_t size, bool inverse) {
    if (size < 2)
        return;
    const uint32_t c = size / 2;
    // forward: out[k] = in[(k - c) mod size] (roll by floor(size/2)); inverse undoes it
    const uint32_t rot = inverse ? (size - c) : c;
    T* tmp = (T*)malloc(sizeof(T) * size);
    if (!tmp)
        return;
    for (uint32_t k = 0; k < size; ++k)
        tmp[(k + rot) % size] = buf[k];
    memcpy(buf, tmp, sizeof(T) * size);
    free(tmp);
}

// Device buffers: one 2D roll on the GPU (in place when every dimension is even
// or 1, else a gather through `tmp`, or through a temporary when tmp is not
// device memory), synchronous like the host path.
template <typename T>
static void shift_dev(T* buf, T* tmp, uint32_t x, uint32_t y, bool inverse) {
    hipStream_t s = entry_stream();
    void* t = nullptr;
    bool own = false;
    if (!shift_in_place(x, y)) {
        if (tmp && is_device_ptr(tmp)) {
            t = tmp;
        } else if (hip_ok(hipMalloc(&t, sizeof(T) * (size_t)x * y), "shift temporary")) {
            own = true;
        } else {
            return;
        }
    }
    (void)hip_ok(launch_shift((int)sizeof(T), buf, t, x, y, inverse, s), "shift");
    (void)hip_ok(hipStreamSynchronize(s), "shift sync");
    if (own)
        (void)hipFree(t);
}

template <typename T>
static void shift_any(T* buf, uint32_t size, bool inverse) {
    if (is_device_ptr(buf)) {
        shift_dev(buf, (T*)nullptr, size, 1, inverse);
        return;
    }
    shift_host(buf, size, inverse);
}

// 2D shift (ext/2d/kfft_cpx2.c:188-240): rows, then columns.
template <typename T>
static void shift2_any(T* buf, T* ftmp, uint32_t x, uint32_t y, bool inverse) {
    if (is_device_ptr(buf)) {
        shift_dev(buf, ftmp, x, y, inverse);
        return;
    }
    for (uint32_t r = 0; r < y; ++r)
        shift_host(buf + (size_t)r * x, x, inverse);
    T* col = (T*)malloc(sizeof(T) * y);
    if (col) {
        for (uint32_t c = 0; c < x; ++c) {
            for (uint32_t r = 0; r < y; ++r)
                col[r] = buf[(size_t)r * x + c];
            shift_host(col, y, inverse);
            for (uint32_t r = 0; r < y; ++r)
                buf[(size_t)r * x + c] = col[r];
        }
        free(col);
    }
}


// In-place transposes (kfft_math.c:80-121): the result is the out-of-place
// transpose written over the input; device buffers go through a temporary.
template <typename T>
static void transpose_ip_any(T* buf, uint32_t x, uint32_t y) {
    if (x <= 1 || y <= 1)
        return;
    const size_t n = (size_t)x * y;
    if (is_device_ptr(buf)) {
        hipStream_t s = entry_stream();
        void* t = nullptr;
        if (!hip_ok(hipMalloc(&t, sizeof(T) * n), "transpose temporary"))
            return;
        if (hip_ok(launch_transpose((int)sizeof(T), buf, t, x, y, 1, s), "transpose"))
            (void)hip_ok(hipMemcpyAsync(buf, t, sizeof(T) * n, hipMemcpyDeviceToDevice, s),
                         "transpose copy");
        (void)hip_ok(hipStreamSynchronize(s), "transpose sync");
        (void)hipFree(t);
        return;
    }
    T* t = (T*)malloc(sizeof(T) * n);
    if (!t)
        return;
    memcpy(t, buf, sizeof(T) * n);
    for (uint64_t k = 0; k < (uint64_t)n; k++)
        buf[k] = t[(uint64_t)x * (k % y) + k / y];
    free(t);
}

// ====================================================================== API
extern "C" {

// ---------------------------------------------------------------- service
KFFT_API void kfft_info(kfft_info_t* info) {
    if (!info)
        return;
    info->vmajor = KFFT_MAJOR_VERSION;
    info->vminor = KFFT_MINOR_VERSION;
    info->vpatch = KFFT_PATCH_VERSION;
    info->flags = KFFT_INFO_RADER_ALGO | KFFT_INFO_GPU_HIP;
#if defined(KFFT_HALF_SCALAR)
    info->flags |= KFFT_INFO_HALF_SCALAR;
#endif
}

KFFT_API uint32_t kfft_next_fast_size(uint32_t n) {
    for (;; n++) {
        uint32_t m = n;
        while (m % 2 == 0)
            m /= 2;
        while (m % 3 == 0)
            m /= 3;
        while (m % 5 == 0)
            m /= 5;
        if (m <= 1)
            return n;
    }
}

KFFT_API void* kfft_malloc(uint32_t sz) { return aligned_alloc(64, ((size_t)sz + 63) / 64 * 64); }

KFFT_API void kfft_free_null(void** mem) {
    if (!mem)
        return;
    free(*mem);
    *mem = nullptr;
}

KFFT_API kfft_return_t kfft_cleanup(void* mem) {
    if (!mem)
        return KFFT_RET_FREE_NULL;
    kfft_object_t* M = (kfft_object_t*)mem;
    if (M->mmgr == nullptr)
        return KFFT_RET_FREE_NULL;
    kfft_pool_free(M->mmgr);
    return KFFT_RET_SUCCESS;
}

KFFT_API const char* kfft_strerr(const kfft_return_t code) {
    static const char* msgs[] = {"Success operation result",
                                 "Internal allocation memory fail",
                                 "Temporary buffer allocation fail",
                                 "Invalide free() operation for NULL buffer",
                                 "Use improper real function for this plan",
                                 "Use missing argument for configure plan",
                                 "GPU operation failed (see kfft_gpu_last_error)"};
    return code < sizeof(msgs) / sizeof(msgs[0]) ? msgs[code] : "Unknown error";
}

// ---------------------------------------------------------------- complex
KFFT_API kfft_plan_cpx* kfft_config_cpx(const uint32_t nfft, const uint32_t flags, kfft_pool_t* A,
                                        size_t* lenmem) {
    return config_cpx(nfft, flags, A, lenmem);
}

KFFT_API kfft_return_t kfft_eval_cpx(kfft_plan_cpx* plan, const kfft_cpx* fin, kfft_cpx* fout) {
    return cpx_run(plan, fin, fout, 1);
}

// ----------------------------------------------------------------- scalar
KFFT_API kfft_plan_sclr* kfft_config_scalar(const uint32_t nfft, const uint32_t flags,
                                            kfft_pool_t* A, size_t* lenmem) {
    return config_sclr(nfft, flags, A, lenmem);
}
KFFT_API kfft_return_t kfft_eval_scalar(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                        kfft_cpx* fout) {
    return sclr_fwd(plan, fin, fout, 1);
}
KFFT_API kfft_return_t kfft_evali_scalar(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                         kfft_scalar* fout) {
    return sclr_inv(plan, fin, fout, 1);
}
KFFT_API kfft_return_t kfft_eval_scalar_internal(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                                 kfft_cpx* fout, kfft_cpx* ftmp) {
    (void)ftmp;
    return sclr_fwd(plan, fin, fout, 1);
}
KFFT_API kfft_return_t kfft_evali_scalar_internal(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                                  kfft_scalar* fout, kfft_cpx* ftmp) {
    (void)ftmp;
    return sclr_inv(plan, fin, fout, 1);
}

// --------------------------------------------------------------------- 2D
KFFT_API kfft_plan_c2d* kfft_config2_cpx(const uint32_t x_size, const uint32_t y_size,
                                         const uint32_t flags, kfft_pool_t* A, size_t* lenmem) {
    return config2_cpx(x_size, y_size, flags, A, lenmem);
}
KFFT_API kfft_return_t kfft_eval2_cpx(kfft_plan_c2d* cfg, const kfft_cpx* fin, kfft_cpx* fout) {
    return c2d_run(cfg, fin, fout);
}

KFFT_API kfft_plan_s2d* kfft_config2_scalar(const uint32_t x_size, const uint32_t y_size,
                                            const uint32_t flags, kfft_pool_t* A,
                                            size_t* lenmem) {
    return config2_sclr(x_size, y_size, flags, A, lenmem);
}

KFFT_API kfft_return_t kfft_eval2_scalar(kfft_plan_s2d* plan, const kfft_scalar* fin,
                                         kfft_cpx* fout) {
    if (!plan || !fin || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    if (plan->flags & KFFT_FLAG_INVERSE)
        return KFFT_RET_IMPROPER_PLAN;
    S2dObj* g = (S2dObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    Staged si, so;
    if (!stage_in(fin, (size_t)plan->nfft * sizeof(kfft_scalar), g->stage_in, si, s) ||
        !stage_out(fout, (size_t)plan->nfft * CPXB, g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = s2d_fwd_dev(plan, si.dev, (void*)so.dev, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_return_t kfft_evali2_scalar(kfft_plan_s2d* plan, const kfft_cpx* fin,
                                          kfft_scalar* fout) {
    if (!plan || !fin || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    if (!(plan->flags & KFFT_FLAG_INVERSE))
        return KFFT_RET_IMPROPER_PLAN;
    S2dObj* g = (S2dObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    Staged si, so;
    if (!stage_in(fin, (size_t)plan->nfft * CPXB, g->stage_in, si, s) ||
        !stage_out(fout, (size_t)plan->nfft * sizeof(kfft_scalar), g->stage_out, so))
        return gpu_fail("staging");
    kfft_return_t r = s2d_inv_dev(plan, si.dev, (void*)so.dev, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

// ------------------------------------------------------------ convolution
// FFT(A), FFT(B) with the forward plan, pointwise product, inverse plan
// (ext/conv/kfft_cpx_conv.c:75-104); the product is fused into the inverse
// transform's load where the inverse is a one- or two-pass transform.
KFFT_API kfft_plan_ccnv* kfft_config_conv_cpx(const uint32_t nfft, const uint32_t flags,
                                              kfft_pool_t* A, size_t* lenmem) {
    const size_t need = sizeof(kfft_plan_ccnv) + 2 * cpx_plan_bytes(nfft);
    kfft_plan_ccnv* P = plan_prepare<kfft_plan_ccnv>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = nfft;
    P->flags = flags;
    const uint32_t f = KFFT_CHECK_FLAGS_CCNV(flags);
    P->plan_fwd = config_cpx(nfft, f, mm, nullptr);
    P->plan_inv = config_cpx(nfft, f | KFFT_FLAG_INVERSE, mm, nullptr);
    ConvObj* g = (P->plan_fwd && P->plan_inv) ? new (std::nothrow) ConvObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

KFFT_API kfft_return_t kfft_eval_conv_cpx(kfft_plan_ccnv* plan, const kfft_cpx* fin_A,
                                          const kfft_cpx* fin_B, kfft_cpx* fout) {
    if (!plan || !fin_A || !fin_B || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    ConvObj* g = (ConvObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    const uint32_t n = plan->nfft;
    const size_t bytes = (size_t)n * CPXB;
    Staged sa, sb, so;
    if (!stage_in(fin_A, bytes, g->stage_in, sa, s) || !stage_in(fin_B, bytes, g->stage_in2, sb, s) ||
        !stage_out(fout, bytes, g->stage_out, so) || !g->work_a.ensure(bytes) ||
        !g->work_b.ensure(bytes))
        return gpu_fail("staging");
    const Plan1D& pf = *((CpxObj*)plan->plan_fwd->gpu)->p;
    if (!g->scratch.ensure(pf.scratch_bytes(1)))
        return gpu_fail("scratch");
    hipError_t e = pf.execute(contiguous(sa.dev, n), contiguous(g->work_a.p, n), 1, false, 1.0,
                              g->scratch.p, s);
    if (e == hipSuccess)
        e = pf.execute(contiguous(sb.dev, n), contiguous(g->work_b.p, n), 1, false, 1.0,
                       g->scratch.p, s);
    if (!hip_ok(e, "conv forward"))
        return KFFT_RET_GPU_FAIL;
    const double sc = cpx_scale(plan->plan_inv);
    if (pf.kind() == Kind::Direct || pf.kind() == Kind::Identity) {
        Fuse fz;
        fz.pw_in = g->work_a.p;
        e = pf.execute(contiguous(g->work_b.p, n), contiguous(so.dev, n), 1, true, sc, g->scratch.p,
                       s, &fz);
    } else {
        hadamard_dev(g->work_b.p, g->work_a.p, n, s);
        e = pf.execute(contiguous(g->work_b.p, n), contiguous(so.dev, n), 1, true, sc, g->scratch.p,
                       s);
    }
    if (!hip_ok(e, "conv inverse"))
        return KFFT_RET_GPU_FAIL;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_plan_scnv* kfft_config_conv_scalar(const uint32_t nfft, const uint32_t flags,
                                                 kfft_pool_t* A, size_t* lenmem) {
    const size_t need = sizeof(kfft_plan_scnv) + 2 * sclr_plan_bytes(nfft);
    kfft_plan_scnv* P = plan_prepare<kfft_plan_scnv>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = nfft;
    P->flags = flags;
    const uint32_t f = KFFT_CHECK_FLAGS(flags) & ~(uint32_t)KFFT_FLAG_INVERSE;
    P->plan_fwd = config_sclr(nfft, f, mm, nullptr);
    P->plan_inv = config_sclr(nfft, f | KFFT_FLAG_INVERSE, mm, nullptr);
    ConvObj* g = (P->plan_fwd && P->plan_inv) ? new (std::nothrow) ConvObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

// ext/conv/kfft_scalar_conv.c:74-100: real forward of both inputs, product
// over the stored spectrum, real inverse (x2 for even n, as the reference).
KFFT_API kfft_return_t kfft_eval_conv_scalar(kfft_plan_scnv* plan, const kfft_scalar* fin_A,
                                             const kfft_scalar* fin_B, kfft_scalar* fout) {
    if (!plan || !fin_A || !fin_B || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    ConvObj* g = (ConvObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    const uint32_t n = plan->nfft, ol = sclr_out_len(plan->plan_fwd);
    const size_t rb = (size_t)n * sizeof(kfft_scalar), cb = (size_t)ol * CPXB;
    Staged sa, sb, so;
    if (!stage_in(fin_A, rb, g->stage_in, sa, s) || !stage_in(fin_B, rb, g->stage_in2, sb, s) ||
        !stage_out(fout, rb, g->stage_out, so) || !g->work_a.ensure(cb) || !g->work_b.ensure(cb))
        return gpu_fail("staging");
    kfft_return_t r = sclr_fwd_dev(plan->plan_fwd, sa.dev, g->work_a.p, 1, ol,
                                   (plan->plan_fwd->flags & KFFT_FLAG_EXPAND_SCALAR) != 0, s);
    if (r == KFFT_RET_SUCCESS)
        r = sclr_fwd_dev(plan->plan_fwd, sb.dev, g->work_b.p, 1, ol,
                         (plan->plan_fwd->flags & KFFT_FLAG_EXPAND_SCALAR) != 0, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    // the product rides on the inverse's first read (its pre-pass, or the load
    // of its one complex pass for odd n)
    r = sclr_inv_dev(plan->plan_inv, g->work_b.p, ol, (void*)so.dev, 1, s, g->work_a.p);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

// ext/conv2d/kfft_cpx_conv.c: the reference builds x-by-x plans (plan->y = x
// at :67), which is a true 2D convolution only for square inputs; this
// library computes the x-by-y convolution for every shape.
KFFT_API kfft_plan_c2cnv* kfft_config2_conv_cpx(const uint32_t x, const uint32_t y,
                                                const uint32_t flags, kfft_pool_t* A,
                                                size_t* lenmem) {
    const size_t need = sizeof(kfft_plan_c2cnv) + 2 * c2d_plan_bytes(x, y);
    kfft_plan_c2cnv* P = plan_prepare<kfft_plan_c2cnv>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = x * y;
    P->x = x;
    P->y = y;
    P->flags = flags;
    const uint32_t f = KFFT_CHECK_FLAGS_CCNV(flags);
    P->plan_fwd = config2_cpx(x, y, f, mm, nullptr);
    P->plan_inv = config2_cpx(x, y, f | KFFT_FLAG_INVERSE, mm, nullptr);
    ConvObj* g = (P->plan_fwd && P->plan_inv) ? new (std::nothrow) ConvObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    return P;
}

KFFT_API kfft_return_t kfft_eval2_conv_cpx(kfft_plan_c2cnv* plan, const kfft_cpx* fin_A,
                                           const kfft_cpx* fin_B, kfft_cpx* fout) {
    if (!plan || !fin_A || !fin_B || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    ConvObj* g = (ConvObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    const size_t bytes = (size_t)plan->nfft * CPXB;
    Staged sa, sb, so;
    if (!stage_in(fin_A, bytes, g->stage_in, sa, s) || !stage_in(fin_B, bytes, g->stage_in2, sb, s) ||
        !stage_out(fout, bytes, g->stage_out, so) || !g->work_a.ensure(bytes) ||
        !g->work_b.ensure(bytes))
        return gpu_fail("staging");
    kfft_return_t r = c2d_run_dev(plan->plan_fwd, sa.dev, g->work_a.p, s);
    if (r == KFFT_RET_SUCCESS)
        r = c2d_run_dev(plan->plan_fwd, sb.dev, g->work_b.p, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    // the product rides on the inverse rows' load where their plan allows
    const Plan1D& pxi = *((CpxObj*)plan->plan_inv->plan_x->gpu)->p;
    const bool fuse = rows_take_product(pxi);
    if (!fuse)
        hadamard_dev(g->work_b.p, g->work_a.p, plan->nfft, s);
    r = c2d_run_dev(plan->plan_inv, g->work_b.p, (void*)so.dev, s, fuse ? g->work_a.p : nullptr);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_plan_s2cnv* kfft_config2_conv_scalar(const uint32_t x, const uint32_t y,
                                                   const uint32_t flags, kfft_pool_t* A,
                                                   size_t* lenmem) {
    const uint32_t f = KFFT_CHECK_FLAGS(flags) & ~(uint32_t)KFFT_FLAG_INVERSE;
    const size_t need = sizeof(kfft_plan_s2cnv) + s2d_plan_bytes(x, y, f) +
                        s2d_plan_bytes(x, y, f | KFFT_FLAG_INVERSE);
    kfft_plan_s2cnv* P = plan_prepare<kfft_plan_s2cnv>(flags, need, A, lenmem);
    if (!P)
        return nullptr;
    kfft_pool_t* mm = P->object.mmgr;
    P->nfft = x * y;
    P->x = x;
    P->y = y;
    P->flags = flags;
    P->plan_fwd = config2_sclr(x, y, f, mm, nullptr);
    P->plan_inv = config2_sclr(x, y, f | KFFT_FLAG_INVERSE, mm, nullptr);
    ConvObj* g = (P->plan_fwd && P->plan_inv) ? new (std::nothrow) ConvObj() : nullptr;
    if (!g) {
        plan_terminate(P, A);
        return nullptr;
    }
    pool_register(mm, g);
    P->gpu = g;
    // the half-spectrum form needs an inverse real plan of the width (even
    // widths); without one the evaluation takes the full-spectrum form
    if (x % 2 == 0)
        g->rows_inv = config_sclr(x, f | KFFT_FLAG_INVERSE, nullptr, nullptr);
    if (g->rows_inv)
        (void)g->cols.plan(y, PREC); // (not compiled, or no table: separate column passes)
    return P;
}

// Real conv2d over the Hermitian-independent half of the spectrum (even x).
// The reference transforms both inputs to full x-by-y spectra (real rows
// expanded, complex columns), multiplies them and inverts with complex rows
// then real columns (ext/conv2d/kfft_scalar_conv.c:92-98,
// ext/2d/kfft_scalar2.c:109-148, 195-226).  Both spectra are Hermitian, so
// columns 0..x/2 hold all of it: here real rows keep x/2+1 bins, the columns
// run over those only, the product rides on the inverse columns' load, and
// real inverse rows (bins 0..x/2) give the output.  The scale reproduces the
// reference's: its real inverse of an even length m returns 2x the normalised
// inverse (1 / (m/2) on a spectrum rebuilt without the halving), so
//   reference: rows 1/x, columns c_y  ->  c_y  x normalised inverse
//   here:      columns s, rows c_x=2  ->  s y c_x x normalised inverse
// with c_y = 2 (even y) or 1 (odd y), giving s = c_y / (2 y); unnormalised
// (KFFT_FLAG_DISABLE_NORM) both are the plain unnormalised inverse (s = 1).
static kfft_return_t conv2_real_half(kfft_plan_s2cnv* plan, ConvObj* g, const void* da,
                                     const void* db, void* dout, hipStream_t s) {
    const uint32_t x = plan->x, y = plan->y, w = x / 2 + 1;
    kfft_plan_s2d* pf = plan->plan_fwd;
    kfft_plan_sclr* sx = (kfft_plan_sclr*)pf->plan_x;
    kfft_plan_cpx* cy = (kfft_plan_cpx*)pf->plan_y;
    const Plan1D& py = *((CpxObj*)cy->gpu)->p;
    const bool unnorm = (plan->plan_inv->flags & KFFT_FLAG_DISABLE_NORM) != 0;
    const double col_scale = unnorm ? 1.0 : ((y % 2) ? 1.0 : 2.0) / (2.0 * y);
    // columns in one pass where their length is compiled and there are enough of them
    // (the split forms run every transform through their own passes).  Rows whose rebuild
    // is in their store leave their spectra in blocks of four columns: a column tile's
    // accesses then share their lines with the next rows' (a 4160-row FP32 tile of two columns
    // reads 16 bytes a row); other rows start on 128-byte lines.
    bool fused = g->cols.y == y && colconv_wide(y, PREC, w) && !split_dft_default();
    bool blk4 = fused && sclr_fuses_blocked(sx);
    uint32_t pitch = blk4 ? (w + 3) / 4 * 4 : fused ? (w + 15) / 16 * 16 : w;
    size_t hb = (size_t)pitch * y * CPXB;
    if (!g->work_a.ensure(hb) || !g->work_b.ensure(hb)) {
        // (no room for the columns past the last: separate passes on exact rows)
        fused = blk4 = false;
        pitch = w;
        hb = (size_t)pitch * y * CPXB;
        if (!g->work_a.ensure(hb) || !g->work_b.ensure(hb))
            return gpu_fail("work");
    }
    const void* in[2] = {da, db};
    DevBuf* spec[2] = {&g->work_a, &g->work_b};
    for (int i = 0; i < 2; ++i) {
        kfft_return_t r = sclr_fwd_dev(sx, in[i], spec[i]->p, y, pitch, false, s, blk4);
        if (r == KFFT_RET_SUCCESS && !fused)
            r = cols_cpx_dev(py, spec[i]->p, w, y, 1, false, 1.0, g->scratch, g->work_c, s);
        if (r != KFFT_RET_SUCCESS)
            return r;
    }
    if (fused) {
        if (!hip_ok(g->cols.run(g->work_a.p, g->work_b.p, blk4, pitch, w, col_scale, s),
                    "conv2d columns"))
            return KFFT_RET_GPU_FAIL;
    } else if (rows_take_product(py) && !py.two_pass() && py.supports_plain_columns()) {
        if (!g->scratch.ensure(py.scratch_bytes(w)))
            return gpu_fail("scratch");
        Layout l;
        l.ptr = g->work_b.p;
        l.C = w;
        l.dist_hi = (int64_t)w * y;
        l.dist_lo = 1;
        l.stride = w;
        Fuse fz;
        fz.pw_in = g->work_a.p;
        hipError_t e = py.execute(l, l, w, true, col_scale, g->scratch.p, s, &fz);
        if (!hip_ok(e, "conv2d inverse columns"))
            return KFFT_RET_GPU_FAIL;
    } else {
        hadamard_dev(g->work_b.p, g->work_a.p, (uint64_t)w * y, s);
        kfft_return_t r =
            cols_cpx_dev(py, g->work_b.p, w, y, 1, true, col_scale, g->scratch, g->work_c, s);
        if (r != KFFT_RET_SUCCESS)
            return r;
    }
    return sclr_inv_dev(g->rows_inv, g->work_b.p, pitch, dout, y, s, nullptr, blk4);
}

KFFT_API kfft_return_t kfft_eval2_conv_scalar(kfft_plan_s2cnv* plan, const kfft_scalar* fin_A,
                                              const kfft_scalar* fin_B, kfft_scalar* fout) {
    if (!plan || !fin_A || !fin_B || !fout || !plan->gpu)
        return KFFT_RET_BADARGUMENTS;
    ConvObj* g = (ConvObj*)plan->gpu;
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = entry_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    const size_t rb = (size_t)plan->nfft * sizeof(kfft_scalar), cb = (size_t)plan->nfft * CPXB;
    Staged sa, sb, so;
    if (!stage_in(fin_A, rb, g->stage_in, sa, s) || !stage_in(fin_B, rb, g->stage_in2, sb, s) ||
        !stage_out(fout, rb, g->stage_out, so))
        return gpu_fail("staging");
    if (g->rows_inv) {
        kfft_return_t r = conv2_real_half(plan, g, sa.dev, sb.dev, (void*)so.dev, s);
        if (r != KFFT_RET_SUCCESS)
            return r;
        return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                              : KFFT_RET_GPU_FAIL;
    }
    if (!g->work_a.ensure(cb) || !g->work_b.ensure(cb))
        return gpu_fail("work");
    kfft_return_t r = s2d_fwd_dev(plan->plan_fwd, sa.dev, g->work_a.p, s);
    if (r == KFFT_RET_SUCCESS)
        r = s2d_fwd_dev(plan->plan_fwd, sb.dev, g->work_b.p, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    hadamard_dev(g->work_b.p, g->work_a.p, plan->nfft, s);
    r = s2d_inv_dev(plan->plan_inv, g->work_b.p, (void*)so.dev, s);
    if (r != KFFT_RET_SUCCESS)
        return r;
    return (finish_out(so, s) && order.sync()) ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}

// ------------------------------------------------------------------- SIMD
// simd/kfft_simd_check.c:132-175.  The host CPU's extensions, as cpuid reports
// them; the build itself uses none (its transforms run on the GPU).
KFFT_API kfft_simd_t kfft_simd_analize(void) {
    kfft_simd_t S = {0, 0};
#if (defined(__x86_64__) || defined(__i386__)) && !defined(__HIP_DEVICE_COMPILE__)
    S.arch = sizeof(void*) == 8 ? HW_ARCH_X64 : HW_ARCH_X86;
    __builtin_cpu_init();
    uint32_t e = sizeof(void*) == 8 ? HW_x64 : 0u;
    e |= __builtin_cpu_supports("mmx") ? HW_MMX : 0u;
    e |= __builtin_cpu_supports("popcnt") ? HW_ABM : 0u;
    e |= __builtin_cpu_supports("bmi") ? HW_BMI1 : 0u;
    e |= __builtin_cpu_supports("bmi2") ? HW_BMI2 : 0u;
    e |= __builtin_cpu_supports("sse") ? HW_SSE : 0u;
    e |= __builtin_cpu_supports("sse2") ? HW_SSE2 : 0u;
    e |= __builtin_cpu_supports("sse3") ? HW_SSE3 : 0u;
    e |= __builtin_cpu_supports("ssse3") ? HW_SSSE3 : 0u;
    e |= __builtin_cpu_supports("sse4.1") ? HW_SSE41 : 0u;
    e |= __builtin_cpu_supports("sse4.2") ? HW_SSE42 : 0u;
    e |= __builtin_cpu_supports("sse4a") ? HW_SSE4a : 0u;
    e |= __builtin_cpu_supports("aes") ? HW_AES : 0u;
    e |= __builtin_cpu_supports("avx") ? HW_AVX : 0u;
    e |= __builtin_cpu_supports("xop") ? HW_XOP : 0u;
    e |= __builtin_cpu_supports("fma") ? HW_FMA3 : 0u;
    e |= __builtin_cpu_supports("fma4") ? HW_FMA4 : 0u;
    e |= __builtin_cpu_supports("avx2") ? HW_AVX2 : 0u;
    e |= __builtin_cpu_supports("avx512f") ? HW_AVX512_F : 0u;
    e |= __builtin_cpu_supports("avx512cd") ? HW_AVX512_CD : 0u;
    e |= __builtin_cpu_supports("avx512vl") ? HW_AVX512_VL : 0u;
    e |= __builtin_cpu_supports("avx512bw") ? HW_AVX512_BW : 0u;
    e |= __builtin_cpu_supports("avx512dq") ? HW_AVX512_DQ : 0u;
    e |= __builtin_cpu_supports("avx512ifma") ? HW_AVX512_IFMA : 0u;
    e |= __builtin_cpu_supports("avx512vbmi") ? HW_AVX512_VBMI : 0u;
    S.ext = e;
#elif defined(__aarch64__) || defined(__arm__)
    S.arch = HW_ARCH_ARM;
#endif
    return S;
}

KFFT_API kfft_simd_t kfft_simd_info(void) {
    kfft_simd_t S = {0, 0};
#if defined(__x86_64__)
    S.arch = HW_ARCH_X64;
#elif defined(__i386__)
    S.arch = HW_ARCH_X86;
#elif defined(__aarch64__) || defined(__arm__)
    S.arch = HW_ARCH_ARM;
#endif
    return S;
}

// ------------------------------------------------------------------- math
KFFT_API void kfft_math_hadamard_cpx(kfft_cpx* Fout, const kfft_cpx* Fin, uint32_t size) {
    if (is_device_ptr(Fout) && is_device_ptr(Fin)) {
        hipStream_t s = entry_stream();
        hadamard_dev(Fout, Fin, size, s);
        (void)hipStreamSynchronize(s);
        return;
    }
    for (uint32_t i = 0; i < size; i++) {
        const kfft_cpx a = Fout[i], b = Fin[i];
        Fout[i].r = a.r * b.r - a.i * b.i;
        Fout[i].i = a.r * b.i + a.i * b.r;
    }
}

KFFT_API void kfft_math_hadamard_scalar(kfft_scalar* Fout, const kfft_scalar* Fin, uint32_t size) {
    if (is_device_ptr(Fout) && is_device_ptr(Fin)) {
        hipStream_t s = entry_stream();
        (void)hip_ok(launch_hadamard_real(PREC, Fout, Fin, size, s), "hadamard");
        (void)hipStreamSynchronize(s);
        return;
    }
    for (uint32_t i = 0; i < size; i++)
        Fout[i] *= Fin[i];
}

// kfft_math.c:60-78: Fout[i*y + j] = Fin[j*x + i]
KFFT_API void kfft_math_transpose_cpx(const kfft_cpx* Fin, kfft_cpx* Fout, const uint32_t x,
                                      const uint32_t y) {
    if (is_device_ptr(Fin) && is_device_ptr(Fout)) {
        hipStream_t s = entry_stream();
        (void)hip_ok(launch_transpose((int)CPXB, Fin, Fout, x, y, 1, s), "transpose");
        (void)hipStreamSynchronize(s);
        return;
    }
    for (uint64_t n = 0; n < (uint64_t)x * y; n++)
        Fout[n] = Fin[(uint64_t)x * (n % y) + n / y];
}

KFFT_API void kfft_math_transpose_scalar(const kfft_scalar* Fin, kfft_scalar* Fout,
                                         const uint32_t x, const uint32_t y) {
    if (is_device_ptr(Fin) && is_device_ptr(Fout)) {
        hipStream_t s = entry_stream();
        (void)hip_ok(launch_transpose((int)sizeof(kfft_scalar), Fin, Fout, x, y, 1, s), "transpose");
        (void)hipStreamSynchronize(s);
        return;
    }
    for (uint64_t n = 0; n < (uint64_t)x * y; n++)
        Fout[n] = Fin[(uint64_t)x * (n % y) + n / y];
}

KFFT_API void kfft_math_transpose_ip_cpx(kfft_cpx* Fin, const uint32_t x, const uint32_t y) {
    transpose_ip_any(Fin, x, y);
}
KFFT_API void kfft_math_transpose_ip_scalar(kfft_scalar* Fin, const uint32_t x, const uint32_t y) {
    transpose_ip_any(Fin, x, y);
}

// kfft_math.c:123-130: Fout[i] = |Fin[i]|, with a correctly rounded square root
// where the reference's default build bisects to an absolute 5e-4
KFFT_API void kfft_math_magnitude(const kfft_cpx* Fin, kfft_scalar* Fout, uint32_t size) {
    if (is_device_ptr(Fin) && is_device_ptr(Fout)) {
        hipStream_t s = entry_stream();
        (void)hip_ok(launch_magnitude(PREC, Fin, Fout, size, s), "magnitude");
        (void)hip_ok(hipStreamSynchronize(s), "magnitude sync");
        return;
    }
    for (uint32_t i = 0; i < size; i++)
        Fout[i] = std::sqrt(Fin[i].r * Fin[i].r + Fin[i].i * Fin[i].i);
}

// kfft_math.c:132-138: the magnitudes overwrite the first `size` reals of the
// buffer.  Reading element i before writing real i is what the reference's
// loop order gives serially; the GPU computes all magnitudes before any write.
KFFT_API void kfft_math_magnitude_ip(kfft_cpx* Fin, uint32_t size) {
    if (is_device_ptr(Fin)) {
        hipStream_t s = entry_stream();
        void* t = nullptr;
        if (!hip_ok(hipMalloc(&t, sizeof(kfft_scalar) * std::max<uint32_t>(size, 1)),
                    "magnitude temporary"))
            return;
        if (hip_ok(launch_magnitude(PREC, Fin, t, size, s), "magnitude"))
            (void)hip_ok(hipMemcpyAsync(Fin, t, sizeof(kfft_scalar) * size,
                                        hipMemcpyDeviceToDevice, s), "magnitude copy");
        (void)hip_ok(hipStreamSynchronize(s), "magnitude sync");
        (void)hipFree(t);
        return;
    }
    kfft_scalar* out = (kfft_scalar*)Fin;
    for (uint32_t i = 0; i < size; i++) {
        const kfft_cpx v = Fin[i];
        out[i] = std::sqrt(v.r * v.r + v.i * v.i);
    }
}

// kfft_math.c:140-148: the mean of `size` reals, summed in FP64 in a fixed
// order (the reference's OpenMP loop adds into one shared variable without a
// reduction, so its multi-threaded result is not defined; its serial result is
// the plain sum in the build's precision)
KFFT_API kfft_scalar kfft_math_average(const kfft_scalar* Fin, uint32_t size) {
    if (!size)
        return (kfft_scalar)0 / (kfft_scalar)0;
    double acc = 0.0;
    if (is_device_ptr(Fin)) {
        hipStream_t s = entry_stream();
        const uint32_t blocks = (uint32_t)std::min<uint64_t>(1024, (size + 255) / 256);
        double* part = nullptr;
        if (!hip_ok(hipMalloc((void**)&part, sizeof(double) * blocks), "average partials"))
            return (kfft_scalar)0 / (kfft_scalar)0;
        std::vector<double> h(blocks);
        if (hip_ok(launch_partial_sum(PREC, Fin, size, part, blocks, s), "average") &&
            hip_ok(hipMemcpyAsync(h.data(), part, sizeof(double) * blocks,
                                  hipMemcpyDeviceToHost, s), "average copy") &&
            hip_ok(hipStreamSynchronize(s), "average sync"))
            for (double v : h)
                acc += v;
        (void)hipFree(part);
    } else {
        for (uint32_t i = 0; i < size; i++)
            acc += (double)Fin[i];
    }
    return (kfft_scalar)(acc / (double)size);
}

KFFT_API void kfft_shift_cpx(kfft_cpx* buf, const uint32_t size, const bool is_inverse,
                             kfft_pool_t* mmgr) {
    (void)mmgr;
    shift_any(buf, size, is_inverse);
}
KFFT_API void kfft_shift_scalar(kfft_scalar* buf, const uint32_t size, const bool is_inverse,
                                kfft_pool_t* mmgr) {
    (void)mmgr;
    shift_any(buf, size, is_inverse);
}

KFFT_API void kfft_shift2_cpx(kfft_cpx* buf, kfft_cpx* ftmp, const uint32_t sz_x,
                              const uint32_t sz_y, const bool is_inverse, kfft_pool_t* mmgr) {
    (void)mmgr;
    shift2_any(buf, ftmp, sz_x, sz_y, is_inverse);
}
KFFT_API void kfft_shift2_scalar(kfft_scalar* buf, kfft_scalar* ftmp, const uint32_t sz_x,
                                 const uint32_t sz_y, const bool is_inverse, kfft_pool_t* mmgr) {
    (void)mmgr;
    shift2_any(buf, ftmp, sz_x, sz_y, is_inverse);
}

// -------------------------------------------------------------------- GPU
KFFT_API void* kfft_gpu_malloc(size_t bytes) {
    if (!runtime_init())
        return nullptr;
    void* p = nullptr;
    return hip_ok(hipMalloc(&p, bytes), "hipMalloc") ? p : nullptr;
}
KFFT_API void kfft_gpu_free(void* ptr) {
    if (ptr)
        (void)hipFree(ptr);
}
KFFT_API kfft_return_t kfft_gpu_memcpy_h2d(void* dst, const void* src, size_t bytes) {
    return hip_ok(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "h2d") ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}
KFFT_API kfft_return_t kfft_gpu_memcpy_d2h(void* dst, const void* src, size_t bytes) {
    return hip_ok(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "d2h") ? KFFT_RET_SUCCESS
                                                                          : KFFT_RET_GPU_FAIL;
}
KFFT_API kfft_return_t kfft_gpu_synchronize(void) {
    if (!runtime_init())
        return KFFT_RET_GPU_FAIL;
    return hip_ok(hipStreamSynchronize(default_stream()), "sync") ? KFFT_RET_SUCCESS
                                                                 : KFFT_RET_GPU_FAIL;
}
KFFT_API void* kfft_gpu_stream(void) { return runtime_init() ? (void*)default_stream() : nullptr; }

KFFT_API int kfft_gpu_plan_error(const kfft_plan_cpx* plan) {
    if (!plan || !plan->gpu)
        return 0;
    CpxObj* g = dynamic_cast<CpxObj*>((GpuObj*)plan->gpu);
    return (g && g->p) ? g->p->async_error() : 0;
}
KFFT_API const char* kfft_gpu_last_error(void) { return last_error(); }

KFFT_API const char* kfft_gpu_plan_describe(const void* plan) {
    const kfft_plan_cpx* P = (const kfft_plan_cpx*)plan;
    if (!P || !P->gpu)
        return "";
    CpxObj* g = dynamic_cast<CpxObj*>((GpuObj*)P->gpu);
    return (g && g->p) ? g->p->describe((P->flags & KFFT_FLAG_GPU_ONCHIP) != 0) : "";
}

KFFT_API kfft_return_t kfft_eval_cpx_batch(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                           kfft_cpx* fout, uint32_t batch) {
    return cpx_run(plan, fin, fout, batch);
}

KFFT_API kfft_return_t kfft_eval_cpx_batch_async(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                                 kfft_cpx* fout, uint32_t batch, void* stream) {
    if (!plan || !plan->gpu || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    CpxObj* g = (CpxObj*)plan->gpu;
    if (!is_device_ptr(fin) || !is_device_ptr(fout)) {
        set_error("asynchronous evaluation needs device buffers");
        return KFFT_RET_BADARGUMENTS;
    }
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    return cpx_run_dev(plan, fin, fout, batch, s);
}

// ============================================ allocation-free batched eval
// Scratch of kfft_eval_cpx_batch_noalloc: a file-scope device array, held by
// every GPU the library runs on until the process ends.  On the host its name
// is a stand-in, not a device address: kernels get the address that
// hipGetSymbolAddress reports for the current device (noalloc_scratch).
#define KFA_NOALLOC_SCRATCH_BYTES ((size_t)32 << 20)
static __device__ __align__(256) unsigned char scratch[KFA_NOALLOC_SCRATCH_BYTES];

// the array's address on the current device, looked up once per device on the
// first call there (the device current)
static void* noalloc_scratch() {
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static void* ptr[kMaxDevices] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        set_error("kfft_eval_cpx_batch_noalloc: no usable current device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(mu);
    if (!ptr[dev]) {
        void* p = nullptr;
        if (!hip_ok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "scratch symbol address") || !p)
            return nullptr;
        ptr[dev] = p;
    }
    return ptr[dev];
}

KFFT_API kfft_return_t kfft_eval_cpx_batch_noalloc(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                                   kfft_cpx* fout, uint32_t batch, void* stream) {
    if (!plan || !plan->gpu || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    CpxObj* g = (CpxObj*)plan->gpu;
    if (!g->p)
        return KFFT_RET_BADARGUMENTS;
    if (g->p64) {
        set_error("kfft_eval_cpx_batch_noalloc: refinement plans (KFFT_FLAG_GPU_REFINE) need "
                  "buffers of their own");
        return KFFT_RET_BADARGUMENTS;
    }
    if (!is_device_ptr(fin) || !is_device_ptr(fout)) {
        set_error("kfft_eval_cpx_batch_noalloc needs device buffers");
        return KFFT_RET_BADARGUMENTS;
    }
    const size_t need = g->p->scratch_charge(batch);
    if (need > KFA_NOALLOC_SCRATCH_BYTES) {
        set_error("kfft_eval_cpx_batch_noalloc: " + std::to_string(batch) + " transforms of " +
                  std::to_string(plan->nfft) + " points need " + std::to_string(need) +
                  " bytes of scratch, above its " + std::to_string(KFA_NOALLOC_SCRATCH_BYTES) +
                  "-byte limit");
        return KFFT_RET_BADARGUMENTS;
    }
    void* sc = need ? noalloc_scratch() : nullptr;
    if (need && !sc)
        return KFFT_RET_GPU_FAIL;
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    Fuse fz;
    fz.onchip = (plan->flags & KFFT_FLAG_GPU_ONCHIP) != 0;
    fz.dft = split_dft(plan->flags);
    const bool inverse = (plan->flags & KFFT_FLAG_INVERSE) != 0;
    set_no_alloc(true);
    const hipError_t e = run_groups(*g->p, contiguous(fin, plan->nfft),
                                    contiguous(fout, plan->nfft), batch,
                                    g->p->group_within(batch, KFA_NOALLOC_SCRATCH_BYTES), inverse,
                                    cpx_scale(plan), sc, s, &fz);
    set_no_alloc(false);
    return hip_ok(e, "noalloc execute") ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

KFFT_API uint32_t kfft_scalar_out_len(const kfft_plan_sclr* plan) {
    return plan ? sclr_out_len(plan) : 0;
}

KFFT_API kfft_return_t kfft_eval_scalar_batch(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                              kfft_cpx* fout, uint32_t batch) {
    return sclr_fwd(plan, fin, fout, batch);
}
KFFT_API kfft_return_t kfft_evali_scalar_batch(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                               kfft_scalar* fout, uint32_t batch) {
    return sclr_inv(plan, fin, fout, batch);
}
KFFT_API kfft_return_t kfft_eval_scalar_batch_async(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                                    kfft_cpx* fout, uint32_t batch, void* stream) {
    if (!plan || !plan->gpu || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    if (plan->basis->flags & KFFT_FLAG_INVERSE)
        return KFFT_RET_IMPROPER_PLAN;
    SclrObj* g = (SclrObj*)plan->gpu;
    if (!is_device_ptr(fin) || !is_device_ptr(fout)) {
        set_error("asynchronous evaluation needs device buffers");
        return KFFT_RET_BADARGUMENTS;
    }
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    return sclr_fwd_dev(plan, fin, fout, batch, sclr_out_len(plan),
                        (plan->flags & KFFT_FLAG_EXPAND_SCALAR) != 0, s);
}
KFFT_API kfft_return_t kfft_evali_scalar_batch_async(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                                     kfft_scalar* fout, uint32_t batch,
                                                     void* stream) {
    if (!plan || !plan->gpu || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    if (!(plan->basis->flags & KFFT_FLAG_INVERSE))
        return KFFT_RET_IMPROPER_PLAN;
    SclrObj* g = (SclrObj*)plan->gpu;
    if (!is_device_ptr(fin) || !is_device_ptr(fout)) {
        set_error("asynchronous evaluation needs device buffers");
        return KFFT_RET_BADARGUMENTS;
    }
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    return sclr_inv_dev(plan, fin, sclr_out_len(plan), fout, batch, s);
}

KFFT_API kfft_return_t kfft_eval2_cpx_async(kfft_plan_c2d* plan, const kfft_cpx* fin,
                                            kfft_cpx* fout, void* stream) {
    if (!plan || !plan->gpu || !fin || !fout)
        return KFFT_RET_BADARGUMENTS;
    C2dObj* g = (C2dObj*)plan->gpu;
    if (!is_device_ptr(fin) || !is_device_ptr(fout)) {
        set_error("asynchronous evaluation needs device buffers");
        return KFFT_RET_BADARGUMENTS;
    }
    std::lock_guard<std::mutex> lk(g->mu);
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    PlanOrder order(g, s);
    if (!order.ok)
        return KFFT_RET_GPU_FAIL;
    SplitScope split(plan->flags);
    return c2d_run_dev(plan, fin, fout, s);
}

// ----------------------------------------------------------- ragged batch
struct kfft_plan_ragged {
    std::unique_ptr<RaggedPlan> plan;
    std::vector<uint64_t> in_off, out_off;
    uint64_t in_bytes = 0, out_bytes = 0;
    // class -> (count, choice)
    std::map<std::pair<uint32_t, uint32_t>, std::pair<uint32_t, RaggedChoice>> classes;
};

struct kfft_mlp {
    Mlp m;
    std::mutex mu;
    kfft_mlp(uint32_t nin, uint32_t hidden) : m(nin, hidden) {}
};

static std::mutex g_model_mu;
static kfft_mlp* g_model = nullptr;

// Plan shape of every class of a ragged batch (which holds the untuned plan's, its
// default): the cost model's best-ranked applicable choice, or the fastest by
// exhaustive timing when no model is set.
static bool choose_classes(kfft_plan_ragged* R) {
    const std::vector<RaggedChoice> cands = tune_candidates();
    std::lock_guard<std::mutex> lk(g_model_mu);
    if (!g_model) {
        for (auto& kv : R->classes) {
            const uint32_t n = kv.first.first, kind = kv.first.second, cnt = kv.second.first;
            double best = -1;
            for (const RaggedChoice& c : cands) {
                if (!choice_applies(n, kind, PREC, c))
                    continue;
                const double t = tune_measure(n, kind, cnt, PREC, c, 3);
                if (t > 0 && (best < 0 || t < best)) {
                    best = t;
                    kv.second.second = c;
                }
            }
        }
        return true;
    }
    // The timings behind the model, and so its ranking, are throughputs of 2^22 points
    // and more: a smaller batch, whose longest chain of tasks counts, keeps the defaults
    // (400 transforms, 1.6 million points: 0.142 ms, 0.167 with the model's choices)
    uint64_t points = 0;
    for (auto& kv : R->classes)
        points += (uint64_t)kv.first.first * kv.second.first;
    if (points < COST_MIN_POINTS)
        return true;
    // one inference over every (class, applicable choice)
    std::vector<float> X;
    std::vector<std::pair<RaggedChoice*, RaggedChoice>> row;
    for (auto& kv : R->classes)
        for (const RaggedChoice& c : cands) {
            if (!choice_applies(kv.first.first, kv.first.second, PREC, c))
                continue;
            float f[COST_FEATURES];
            cost_features(kv.first.first, kv.first.second, kv.second.first, PREC, c, f);
            X.insert(X.end(), f, f + COST_FEATURES);
            row.push_back({&kv.second.second, c});
        }
    if (row.empty())
        return true;
    std::lock_guard<std::mutex> lm(g_model->mu);
    DevBuf dx, dy;
    std::vector<float> y(row.size());
    hipStream_t s = default_stream();
    if (!dx.alloc(X.size() * 4) || !dy.alloc(y.size() * 4) ||
        !hip_ok(hipMemcpy(dx.p, X.data(), X.size() * 4, hipMemcpyHostToDevice), "model input") ||
        !hip_ok(g_model->m.forward_dev((const float*)dx.p, (float*)dy.p, (uint32_t)row.size(), s),
                "model forward") ||
        !hip_ok(hipStreamSynchronize(s), "model sync") ||
        !hip_ok(hipMemcpy(y.data(), dy.p, y.size() * 4, hipMemcpyDeviceToHost), "model output"))
        return false;
    // leave the default shape unless the model expects a clear gain (its
    // errors are ~10% in time, and classes share the GPU inside a batch)
    std::map<RaggedChoice*, float> best, dflt;
    for (size_t i = 0; i < row.size(); ++i) {
        if (row[i].second == *row[i].first) // (still the class's default)
            dflt[row[i].first] = y[i];
    }
    for (size_t i = 0; i < row.size(); ++i) {
        auto d = dflt.find(row[i].first);
        const float bar = d == dflt.end() ? 1e30f : d->second - COST_MARGIN;
        auto it = best.find(row[i].first);
        if (y[i] < bar && (it == best.end() || y[i] < it->second)) {
            best[row[i].first] = y[i];
            *row[i].first = row[i].second;
        }
    }
    return true;
}

// executor shape, from the environment where set: KFFT_AMD_RAGGED_IPW (largest
// instances per tile), KFFT_AMD_RAGGED_WGS (workgroups per CU),
// KFFT_AMD_RAGGED_LDS (KiB of LDS per workgroup for tiles), KFFT_AMD_RAGGED_GRAPH
// (0: launch directly instead of replaying a captured graph)
static RaggedOptions ragged_options() {
    RaggedOptions o;
    if (const char* e = getenv("KFFT_AMD_RAGGED_IPW"))
        o.ipw_cap = (uint32_t)atoi(e);
    if (const char* e = getenv("KFFT_AMD_RAGGED_WGS"))
        o.wgs_per_cu = (uint32_t)atoi(e);
    if (const char* e = getenv("KFFT_AMD_RAGGED_LDS"))
        o.lds_budget = (uint32_t)atoi(e) * 1024u;
    if (const char* e = getenv("KFFT_AMD_RAGGED_GRAPH"))
        o.graph = atoi(e) != 0;
    return o;
}

KFFT_API kfft_plan_ragged* kfft_config_ragged(uint32_t count, const uint32_t* nfft,
                                              const uint8_t* kind, const uint64_t* in_off,
                                              const uint64_t* out_off, uint32_t flags) {
    if (!count || !nfft || !runtime_init())
        return nullptr;
    std::unique_ptr<kfft_plan_ragged> R(new (std::nothrow) kfft_plan_ragged());
    if (!R)
        return nullptr;
    std::vector<RaggedItem> items(count);
    uint64_t ip = 0, op = 0;
    for (uint32_t i = 0; i < count; ++i) {
        RaggedItem& it = items[i];
        it.n = nfft[i];
        it.kind = kind ? kind[i] : KFFT_RAGGED_COMPLEX;
        const uint64_t in_b = (uint64_t)it.n * (it.kind == KFFT_RAGGED_REAL ? sizeof(kfft_scalar)
                                                                            : CPXB);
        const uint64_t outn = it.kind == KFFT_RAGGED_REAL && it.n % 2 == 0 ? it.n / 2 + 1 : it.n;
        const uint64_t out_b = outn * CPXB;
        it.in_off = in_off ? in_off[i] : ip;
        it.out_off = out_off ? out_off[i] : op;
        ip = (it.in_off + in_b + 255) / 256 * 256;
        op = (it.out_off + out_b + 255) / 256 * 256;
        R->in_bytes = std::max(R->in_bytes, it.in_off + in_b);
        R->out_bytes = std::max(R->out_bytes, it.out_off + out_b);
        R->in_off.push_back(it.in_off);
        R->out_off.push_back(it.out_off);
    }
    const bool inverse = (flags & KFFT_FLAG_INVERSE) != 0;
    for (const RaggedItem& it : items)
        R->classes[{it.n, it.kind}].first++;
    RaggedOptions opt = ragged_options();
    for (auto& kv : R->classes)
        kv.second.second = ragged_default(kv.first.first, kv.first.second, PREC, opt.lds_budget);
    const bool tuned = (flags & KFFT_FLAG_GPU_TUNED) != 0;
    if (tuned) {
        if (inverse) {
            set_error("ragged batch: tuned plans are forward transforms");
            return nullptr;
        }
        if (!choose_classes(R.get()))
            return nullptr;
    }
    kfft_plan_ragged* rp = R.get();
    opt.choose = [rp](uint32_t n, uint32_t kind, uint32_t) {
        return rp->classes[{n, kind}].second;
    };
    R->plan.reset(new (std::nothrow)
                      RaggedPlan(PREC, inverse, !(flags & KFFT_FLAG_DISABLE_NORM)));
    if (!R->plan)
        return nullptr;
    if (!R->plan->build(items, opt)) {
        if (tuned)
            return nullptr;
        // (without room for power-of-two convolution lengths: the shortest ones)
        for (auto& kv : R->classes)
            kv.second.second = RaggedChoice();
        R->plan.reset(new (std::nothrow)
                          RaggedPlan(PREC, inverse, !(flags & KFFT_FLAG_DISABLE_NORM)));
        if (!R->plan || !R->plan->build(items, opt))
            return nullptr;
    }
    return R.release();
}

KFFT_API kfft_return_t kfft_ragged_layout(const kfft_plan_ragged* plan, uint64_t* in_off,
                                          uint64_t* out_off, uint64_t* in_bytes,
                                          uint64_t* out_bytes) {
    if (!plan)
        return KFFT_RET_BADARGUMENTS;
    if (in_off)
        memcpy(in_off, plan->in_off.data(), plan->in_off.size() * 8);
    if (out_off)
        memcpy(out_off, plan->out_off.data(), plan->out_off.size() * 8);
    if (in_bytes)
        *in_bytes = plan->in_bytes;
    if (out_bytes)
        *out_bytes = plan->out_bytes;
    return KFFT_RET_SUCCESS;
}

KFFT_API kfft_return_t kfft_eval_ragged_async(kfft_plan_ragged* plan, const void* in, void* out,
                                              void* stream) {
    if (!plan || !in || !out || !is_device_ptr(in) || !is_device_ptr(out))
        return KFFT_RET_BADARGUMENTS;
    hipStream_t s = stream ? (hipStream_t)stream : default_stream();
    return hip_ok(plan->plan->run(in, out, s), "ragged run") ? KFFT_RET_SUCCESS
                                                             : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_return_t kfft_eval_ragged(kfft_plan_ragged* plan, const void* in, void* out) {
    if (!plan || !in || !out || !is_device_ptr(in) || !is_device_ptr(out))
        return KFFT_RET_BADARGUMENTS;
    hipStream_t s = entry_stream();
    if (!hip_ok(plan->plan->run(in, out, s), "ragged run"))
        return KFFT_RET_GPU_FAIL;
    if (plan->plan->error()) {
        set_error("ragged batch: a dependency wait timed out");
        return KFFT_RET_GPU_FAIL;
    }
    return KFFT_RET_SUCCESS;
}

KFFT_API int kfft_ragged_error(kfft_plan_ragged* plan) { return plan ? plan->plan->error() : 0; }

KFFT_API const char* kfft_ragged_describe(const kfft_plan_ragged* plan) {
    return plan ? plan->plan->describe() : "";
}

KFFT_API void kfft_release_ragged(kfft_plan_ragged* plan) { delete plan; }

KFFT_API uint32_t kfft_ragged_classes(const kfft_plan_ragged* plan, uint32_t* nfft, uint8_t* kind,
                                      uint32_t* count, uint32_t* max_radix, uint32_t* force_four,
                                      uint32_t* ipw_cap) {
    if (!plan)
        return 0;
    uint32_t i = 0;
    for (const auto& kv : plan->classes) {
        if (nfft)
            nfft[i] = kv.first.first;
        if (kind)
            kind[i] = (uint8_t)kv.first.second;
        if (count)
            count[i] = kv.second.first;
        if (max_radix)
            max_radix[i] = kv.second.second.v.maxr;
        if (force_four)
            force_four[i] = (kv.second.second.v.four ? 1u : 0u) | (kv.second.second.v.pow2_m ? 2u : 0u);
        if (ipw_cap)
            ipw_cap[i] = kv.second.second.ipw_cap;
        ++i;
    }
    return i;
}

// ------------------------------------------------------ autotuner, cost model
static RaggedChoice make_choice(uint32_t max_radix, uint32_t force_four, uint32_t ipw_cap) {
    RaggedChoice c;
    c.v.maxr = max_radix >= 16 ? 16u : (max_radix >= 8 ? 8u : 4u);
    c.v.four = (force_four & 1u) != 0;
    c.v.pow2_m = (force_four & 2u) != 0;
    c.ipw_cap = ipw_cap;
    return c;
}

KFFT_API uint32_t kfft_tune_candidates(uint32_t* max_radix, uint32_t* force_four,
                                       uint32_t* ipw_cap) {
    const std::vector<RaggedChoice> c = tune_candidates();
    for (size_t i = 0; i < c.size(); ++i) {
        if (max_radix)
            max_radix[i] = c[i].v.maxr;
        if (force_four)
            force_four[i] = (c[i].v.four ? 1u : 0u) | (c[i].v.pow2_m ? 2u : 0u);
        if (ipw_cap)
            ipw_cap[i] = c[i].ipw_cap;
    }
    return (uint32_t)c.size();
}

KFFT_API double kfft_tune_measure(uint32_t nfft, uint8_t kind, uint32_t count, uint32_t max_radix,
                                  uint32_t force_four, uint32_t ipw_cap, uint32_t reps) {
    if (!runtime_init())
        return -2.0;
    const RaggedChoice c = make_choice(max_radix, force_four, ipw_cap);
    if (!choice_applies(nfft, kind, PREC, c))
        return -1.0;
    return tune_measure(nfft, kind, count, PREC, c, reps);
}

KFFT_API uint32_t kfft_cost_features(uint32_t nfft, uint8_t kind, uint32_t count,
                                     uint32_t max_radix, uint32_t force_four, uint32_t ipw_cap,
                                     float* out) {
    if (out)
        cost_features(nfft, kind, count, PREC, make_choice(max_radix, force_four, ipw_cap), out);
    return (uint32_t)COST_FEATURES;
}

KFFT_API kfft_mlp* kfft_mlp_create(uint32_t nin, uint32_t hidden, uint32_t seed) {
    if (!nin || !hidden || !runtime_init())
        return nullptr;
    std::unique_ptr<kfft_mlp> m(new (std::nothrow) kfft_mlp(nin, hidden));
    if (!m || !m->m.init(seed))
        return nullptr;
    return m.release();
}

KFFT_API uint32_t kfft_mlp_param_count(const kfft_mlp* mlp) {
    return mlp ? mlp->m.param_count() : 0;
}

KFFT_API kfft_return_t kfft_mlp_set_params(kfft_mlp* mlp, const float* host) {
    if (!mlp || !host)
        return KFFT_RET_BADARGUMENTS;
    std::lock_guard<std::mutex> lk(mlp->mu);
    return mlp->m.set_params(host) ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_return_t kfft_mlp_get_params(const kfft_mlp* mlp, float* host) {
    if (!mlp || !host)
        return KFFT_RET_BADARGUMENTS;
    return mlp->m.get_params(host) ? KFFT_RET_SUCCESS : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_return_t kfft_mlp_forward(kfft_mlp* mlp, const float* x, float* y, uint32_t batch) {
    if (!mlp || !x || !y || !batch)
        return KFFT_RET_BADARGUMENTS;
    std::lock_guard<std::mutex> lk(mlp->mu);
    hipStream_t s = entry_stream();
    return hip_ok(mlp->m.forward_dev(x, y, batch, s), "mlp forward") &&
                   hip_ok(hipStreamSynchronize(s), "mlp sync")
               ? KFFT_RET_SUCCESS
               : KFFT_RET_GPU_FAIL;
}

KFFT_API kfft_return_t kfft_mlp_gradient(kfft_mlp* mlp, const float* x, const float* t,
                                         uint32_t batch, float* grad_host, float* loss) {
    if (!mlp || !x || !t || !batch)
        return KFFT_RET_BADARGUMENTS;
    std::lock_guard<std::mutex> lk(mlp->mu);
    hipStream_t s = entry_stream();
    float l = 0.0f;
    if (!hip_ok(mlp->m.gradient_dev(x, t, batch, &l, s), "mlp gradient") ||
        !hip_ok(hipStreamSynchronize(s), "mlp sync") ||
        (grad_host && !mlp->m.get_grads(grad_host)))
        return KFFT_RET_GPU_FAIL;
    if (loss)
        *loss = l;
    return KFFT_RET_SUCCESS;
}

KFFT_API kfft_return_t kfft_mlp_train_step(kfft_mlp* mlp, const float* x, const float* t,
                                           uint32_t batch, float lr, float* loss) {
    if (!mlp || !x || !t || !batch)
        return KFFT_RET_BADARGUMENTS;
    std::lock_guard<std::mutex> lk(mlp->mu);
    hipStream_t s = entry_stream();
    return hip_ok(mlp->m.train_step(x, t, batch, lr, loss, s), "mlp train") ? KFFT_RET_SUCCESS
                                                                           : KFFT_RET_GPU_FAIL;
}

KFFT_API void kfft_mlp_release(kfft_mlp* mlp) {
    std::lock_guard<std::mutex> lk(g_model_mu);
    if (g_model == mlp)
        g_model = nullptr;
    delete mlp;
}

KFFT_API kfft_return_t kfft_ragged_set_cost_model(kfft_mlp* mlp) {
    std::lock_guard<std::mutex> lk(g_model_mu);
    if (mlp && mlp->m.nin() != (uint32_t)COST_FEATURES)
        return KFFT_RET_BADARGUMENTS;
    g_model = mlp;
    return KFFT_RET_SUCCESS;
}

} // extern "C"
