// Planner and executor of the gfx950 transform engine (see kfa_engine.h).
#include "kfa_engine.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "kfa_kernels.h"

namespace kfa {

// ===================================================================== runtime
static thread_local std::string g_err;

void set_error(const std::string& msg) { g_err = msg; }
const char* last_error() { return g_err.c_str(); }

bool hip_ok(hipError_t e, const char* what) {
    if (e == hipSuccess)
        return true;
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return false;
}

static std::mutex g_rt_mu;
static hipStream_t g_stream = nullptr;
static bool g_rt_ready = false;

bool runtime_init() {
    std::lock_guard<std::mutex> lk(g_rt_mu);
    if (g_rt_ready)
        return true;
    int n = 0;
    if (!hip_ok(hipGetDeviceCount(&n), "hipGetDeviceCount"))
        return false;
    if (n <= 0) {
        set_error("no HIP device visible");
        return false;
    }
    if (!hip_ok(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking), "hipStreamCreate"))
        return false;
    g_rt_ready = true;
    return true;
}

hipStream_t default_stream() {
    runtime_init();
    return g_stream;
}

static thread_local bool g_no_alloc = false;
void set_no_alloc(bool on) { g_no_alloc = on; }
bool no_alloc() { return g_no_alloc; }

static thread_local uint32_t g_split_dft = 0;
void set_split_dft(uint32_t dft) { g_split_dft = dft; }
uint32_t split_dft_default() { return g_split_dft; }

// Device bytes the library holds (plans, scratch, staging), and the budget
// KFFT_AMD_DEVICE_LIMIT_MB puts on them (read at every allocation, so a
// process can set or lift it at any time; unset or 0: no budget).  An
// allocation beyond the budget fails like a hipMalloc that runs out of memory.
static std::atomic<size_t> g_dev_bytes{0};

size_t device_bytes_held() { return g_dev_bytes.load(std::memory_order_relaxed); }

size_t device_room() {
    const char* e = getenv("KFFT_AMD_DEVICE_LIMIT_MB");
    const size_t cap = e ? (size_t)strtoull(e, nullptr, 10) << 20 : 0, held = device_bytes_held();
    return !cap ? SIZE_MAX : cap > held ? cap - held : 0;
}

DevBuf::~DevBuf() { release(); }
void DevBuf::release() {
    if (p) {
        // work queued on the library stream or on a caller's stream (the
        // asynchronous entry points) may still read this buffer
        if (g_stream)
            (void)hipDeviceSynchronize();
        (void)hipFree(p);
        g_dev_bytes.fetch_sub(bytes, std::memory_order_relaxed);
    }
    p = nullptr;
    bytes = 0;
}
bool DevBuf::alloc(size_t n) {
    release();
    if (n == 0)
        return true;
    if (n > device_room()) {
        const char* e = getenv("KFFT_AMD_DEVICE_LIMIT_MB");
        set_error("device memory budget (KFFT_AMD_DEVICE_LIMIT_MB=" + std::string(e ? e : "") +
                  ") exceeded: " + std::to_string(n) + " more bytes requested, " +
                  std::to_string(device_bytes_held()) + " held");
        return false;
    }
    if (!hip_ok(hipMalloc(&p, n), "hipMalloc")) {
        (void)hipGetLastError(); // (a caller may go on with less: not the next launch's error)
        p = nullptr;
        return false;
    }
    bytes = n;
    g_dev_bytes.fetch_add(n, std::memory_order_relaxed);
    return true;
}
bool DevBuf::ensure(size_t n) {
    if (n <= bytes)
        return true;
    return alloc(n);
}

bool SharedTab::get(uint32_t kind, uint32_t a, uint32_t b,
                    const std::function<bool(DevBuf&)>& make) {
    static std::mutex mu;
    static std::map<std::tuple<uint32_t, uint32_t, uint32_t>, std::weak_ptr<DevBuf>> tabs;
    std::lock_guard<std::mutex> lk(mu);
    auto& slot = tabs[std::make_tuple(kind, a, b)];
    buf = slot.lock();
    if (!buf) {
        auto n = std::make_shared<DevBuf>();
        // (another thread's plan may use the table as soon as the lock is released)
        if (!make(*n) || !hip_ok(hipStreamSynchronize(default_stream()), "shared table"))
            return false;
        slot = buf = n;
    }
    p = buf->p;
    return true;
}

size_t elem_bytes(int prec) { return 2 * (size_t)prec; }

// ================================================================== LDS passes
static uint32_t pad_index(uint32_t e, int prec) {
    return e + (e >> (prec == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32));
}

std::vector<uint32_t> radix_list(uint32_t L, uint32_t maxr) {
    std::vector<uint32_t> r;
    if (L <= 1)
        return r;
    uint32_t a = 0, b = 0, m = L;
    while (m % 2 == 0) {
        m /= 2;
        ++a;
    }
    while (m % 3 == 0) {
        m /= 3;
        ++b;
    }
    std::vector<uint32_t> odd;
    for (uint32_t p : {5u, 7u, 11u, 13u, 17u, 19u, 23u, 29u, 31u})
        while (m % p == 0) {
            m /= p;
            odd.push_back(p);
        }
    if (m != 1)
        return {};
    if (maxr < 16) {
        // fewer radix-2 levels fused per stage: 8s (or 4s), then the rest
        const uint32_t k = maxr >= 8 ? 3 : 2;
        for (uint32_t i = 0; i < a / k; ++i)
            r.push_back(1u << k);
        if (a % k)
            r.push_back(1u << (a % k));
        for (uint32_t i = 0; i < b; ++i)
            r.push_back(3);
        for (uint32_t p : odd)
            r.push_back(p);
        return r;
    }
    const uint32_t q = a / 4, rr = a % 4;
    // 2^(4q+1): 16s then 8, 4 on the vector units; the split form (maxr =
    // KFA_MAXR_SPLIT) keeps one more radix-16 stage for the matrix cores in
    // the general pass.  Powers of two keep the order of the shaped passes
    // (kfa_fast_impl.h), which share this list's twiddle table.
    const bool pow2 = b == 0 && odd.empty();
    if (rr == 1 && q > 0 && (maxr < KFA_MAXR_SPLIT || pow2)) {
        for (uint32_t i = 0; i + 1 < q; ++i)
            r.push_back(16);
        r.push_back(8);
        r.push_back(4);
    } else {
        for (uint32_t i = 0; i < q; ++i)
            r.push_back(16);
        if (rr == 1)
            r.push_back(2);
        else if (rr == 2)
            r.push_back(4);
        else if (rr == 3)
            r.push_back(8);
    }
    for (uint32_t i = 0; i < b / 2; ++i)
        r.push_back(9);
    if (b % 2)
        r.push_back(3);
    for (uint32_t p : odd)
        r.push_back(p);
    return r;
}

static bool lds_shape(uint32_t L, int prec, int* maxe_out, uint32_t* tpi_out, uint32_t* stride_out,
                      uint32_t maxr = 16) {
    if (L == 1) {
        *maxe_out = 16;
        *tpi_out = 1;
        *stride_out = 1;
        return true;
    }
    std::vector<uint32_t> rl = radix_list(L, maxr);
    if (rl.empty() || rl.size() > KFA_MAX_STAGES)
        return false;
    const uint32_t rmax = *std::max_element(rl.begin(), rl.end());
    const int maxe = rmax > 16 ? 32 : 16;
    uint32_t tpi = 1;
    for (uint32_t R : rl) {
        const uint32_t per = std::max<uint32_t>(1, (uint32_t)maxe / R);
        const uint32_t need = (L / R + per - 1) / per;
        tpi = std::max(tpi, need);
    }
    const uint32_t limit = maxe == 16 ? 512 : 256;
    if (tpi > limit)
        return false;
    uint32_t stride = pad_index(L - 1, prec) + 1;
    stride |= 1u;
    if ((size_t)stride * elem_bytes(prec) > 160 * 1024)
        return false;
    *maxe_out = maxe;
    *tpi_out = tpi;
    *stride_out = stride;
    return true;
}

bool lds_capable(uint32_t L, int prec) {
    int m;
    uint32_t t, s;
    return lds_shape(L, prec, &m, &t, &s);
}

bool LdsPass::plan(uint32_t len, int p, uint32_t max_radix) {
    L = len;
    prec = p;
    if (L >= 65536u) { // the stages' multiply-high modulo needs b, ns < 2^16
        set_error("length " + std::to_string(L) + " is too long for one LDS pass");
        return false;
    }
    if (!lds_shape(L, prec, &maxe, &tpi, &inst_stride, max_radix)) {
        set_error("length " + std::to_string(L) + " does not fit one LDS pass");
        return false;
    }
    return plan_stages(len, p, max_radix);
}

bool LdsPass::plan_stages(uint32_t len, int p, uint32_t max_radix) {
    L = len;
    prec = p;
    std::vector<uint32_t> rl = radix_list(L, max_radix);
    nstages = (uint32_t)rl.size();
    uint32_t ns = 1, off = 0;
    for (uint32_t s = 0; s < nstages; ++s) {
        st[s].radix = rl[s];
        st[s].ns = ns;
        st[s].tw_off = off;
        st[s].ns_magic = ns > 1 ? (uint32_t)(((1ull << 32) + ns - 1) / ns) : 0u;
        if (s > 0)
            off += ns * (rl[s] - 1);
        ns *= rl[s];
    }
    tw_count = nstages >= 2 ? off : 0u;
    if (nstages >= 2) {
        // (a table depends on the radix order, which max_radix and L decide)
        if (!tw.get(prec == 8 ? 0 : 1, L, max_radix, [&](DevBuf& d) {
                KfaFftArgs a;
                memset(&a, 0, sizeof(a));
                a.L = L;
                a.nstages = nstages;
                memcpy(a.st, st, sizeof(st));
                return d.alloc((size_t)std::max<uint32_t>(off, 1) * elem_bytes(prec)) &&
                       hip_ok(launch_stage_twiddles(prec, d.p, a, default_stream()),
                              "stage twiddles");
            }))
            return false;
    }
    return true;
}

uint32_t LdsPass::lds_bytes(uint32_t ipw) const {
    if (nstages == 0 && L <= 1)
        return (uint32_t)(ipw * inst_stride * elem_bytes(prec));
    return (uint32_t)(ipw * inst_stride * elem_bytes(prec));
}

uint32_t LdsPass::pick_ipw(bool jfast) const {
    const uint32_t limit = maxe == 16 ? 512 : 256;
    uint32_t ipw = std::max<uint32_t>(1, 256 / tpi);
    if (jfast)
        ipw = std::max<uint32_t>(ipw, 16);
    while (ipw > 1 && tpi * ipw > limit)
        --ipw;
    const size_t per = (size_t)inst_stride * elem_bytes(prec);
    const size_t budget = 72 * 1024;
    while (ipw > 1 && per * ipw > budget)
        --ipw;
    return ipw;
}

// ==================================================================== SubFft
static bool split_four(uint32_t L, int prec, uint32_t* n1, uint32_t* n2) {
    uint32_t best = 0;
    for (uint32_t d = (uint32_t)std::sqrt((double)L) + 1; d >= 2; --d) {
        if (L % d)
            continue;
        const uint32_t a = std::min(d, L / d), b = std::max(d, L / d);
        if (lds_capable(a, prec) && lds_capable(b, prec)) {
            best = a;
            break;
        }
    }
    if (!best)
        return false;
    *n1 = best;
    *n2 = L / best;
    return true;
}

static uint32_t direct_max(int prec) { return prec == 8 ? 4096u : 8192u; }

// Three passes: L = N1 N2 with a one-pass column length N1 (the smallest from
// 16 on, so that the inner two-pass rows stay long) and a two-pass N2.
static bool split_three(uint32_t L, int prec, uint32_t* n1, uint32_t* n2) {
    uint32_t a, b;
    for (uint32_t lo : {16u, 2u})
        for (uint32_t d = lo; d <= 8192 && d < L; ++d)
            if (L % d == 0 && lds_capable(d, prec) && split_four(L / d, prec, &a, &b)) {
                *n1 = d;
                *n2 = L / d;
                return true;
            }
    return false;
}

bool subfft_capable(uint32_t L, int prec, bool three_ok) {
    if (lds_capable(L, prec))
        return true;
    uint32_t a, b;
    return split_four(L, prec, &a, &b) || (three_ok && split_three(L, prec, &a, &b));
}

// The single-pass 65536-point form runs where a caller asks for the on-chip
// form (KFFT_FLAG_GPU_ONCHIP) and the plan-build probe read the XCD ids.  KFFT_AMD_PAIR=1 makes it the default for
// every eligible call, KFFT_AMD_PAIR=0 turns it off.
static int pair_mode() {
    static const int m = [] {
        const char* e = getenv("KFFT_AMD_PAIR");
        return e ? atoi(e) : -1;
    }();
    return m;
}

static bool shaped_sub(uint32_t N, uint32_t maxr);

// two-level table of W_L^m: S entries W_L^lo and nhi entries W_L^(hi S), FP64
static bool four_step_tables(uint32_t L, uint64_t S, uint64_t nhi, SharedTab& lo, SharedTab& hi) {
    hipStream_t s = default_stream();
    return lo.get(2, L, 0, [&](DevBuf& d) {
        return d.alloc(S * 16) && hip_ok(launch_twiddle_table(d.p, S, 1, L, s), "tw4 lo");
    }) && hi.get(3, L, 0, [&](DevBuf& d) {
        return d.alloc(nhi * 16) && hip_ok(launch_twiddle_table(d.p, nhi, S, L, s), "tw4 hi");
    });
}

// Factors of the inverse real rebuild in pass A's load (kfa_fast_impl.h: rpre_column),
// from long double: W_2N1^n1 and what its rounding left (float), W_2L^n2 - 1.
static bool inverse_rebuild_tables(uint32_t L, uint32_t N1, uint32_t N2, int prec, SharedTab& row,
                                   SharedTab& col) {
    const long double pi = 3.141592653589793238462643383279502884L;
    auto put = [&](std::vector<unsigned char>& b, size_t i, long double v) -> long double {
        if (prec == 8) {
            const double d = (double)v;
            memcpy(&b[i * 8], &d, 8);
            return d;
        }
        const float f = (float)v;
        memcpy(&b[i * 4], &f, 4);
        return f;
    };
    auto table = [&](SharedTab& t, uint32_t kind, auto fill) {
        return t.get(kind + (prec == 8 ? 0u : 1u), L, 0, [&](DevBuf& d) {
            std::vector<unsigned char> b;
            fill(b);
            return d.alloc(b.size()) &&
                   hip_ok(hipMemcpy(d.p, b.data(), b.size(), hipMemcpyHostToDevice),
                          "inverse rebuild factors");
        });
    };
    return table(row, 16, [&](std::vector<unsigned char>& b) {
        const size_t eb = elem_bytes(prec); // (an entry: 2 eb bytes, the low part in its second half)
        b.resize(N1 * 2 * eb);
        for (uint32_t i = 0; i < N1; ++i) {
            const long double a = -pi * i / N1, w[2] = {cosl(a), sinl(a)};
            for (int c = 0; c < 2; ++c) {
                const float lo = (float)(w[c] - put(b, 4 * (size_t)i + c, w[c]));
                memcpy(&b[(2 * (size_t)i + 1) * eb + 4 * c], &lo, 4);
            }
        }
    }) && table(col, 18, [&](std::vector<unsigned char>& b) {
        b.resize(N2 * elem_bytes(prec));
        for (uint32_t i = 0; i < N2; ++i) {
            const long double a = -pi * i / L, s2 = sinl(a / 2);
            put(b, 2 * (size_t)i, -2 * s2 * s2);
            put(b, 2 * (size_t)i + 1, sinl(a));
        }
    });
}

bool SubFft::plan(uint32_t len, int p, bool force_four, uint32_t max_radix) {
    L = len;
    prec = p;
    maxr = max_radix;
    // one pass where it fits: up to direct_max, and every length of the shaped
    // mixed-radix rows (one pass of those beats two general passes)
    const bool mixed_one = mixed_len(L) && maxr == 16;
    if (!force_four && maxr == 16 && bigrow_len(L, prec) && !big.plan_stages(L, prec))
        big = LdsPass(); // (no room for its table: the form below)
    if (!force_four && lds_capable(L, prec) &&
        (L <= direct_max(prec) || mixed_one || !split_four(L, prec, &N1, &N2))) {
        four = false;
        return direct.plan(L, prec, maxr);
    }
    if (!split_four(L, prec, &N1, &N2)) {
        if (force_four || !split_three(L, prec, &N1, &N2)) {
            set_error("length " + std::to_string(L) + " has no two- or three-pass split");
            return false;
        }
        // three passes: the column pass of N1 with W_L^(n2 k1) on its store, then
        // the inner plan's rows
        three = true;
        if (!col.plan(N1, prec, maxr))
            return false;
        inner = get_plan(N2, prec);
        if (!inner)
            return false;
        uint32_t sh = 0;
        while ((1ull << (2 * sh)) < L)
            ++sh;
        tw4_shift = sh;
        const uint64_t S = 1ull << sh, nhi = (L + S - 1) / S + 1;
        return four_step_tables(L, S, nhi, tw4_lo, tw4_hi);
    }
    four = true;
    if (!col.plan(N1, prec, maxr) || !row.plan(N2, prec, maxr))
        return false;
    // two-level table for W_L^m: m = hi*S + lo, S = 2^shift >= sqrt(L)
    uint32_t sh = 0;
    while ((1ull << (2 * sh)) < L)
        ++sh;
    tw4_shift = sh;
    const uint64_t S = 1ull << sh, nhi = (L + S - 1) / S + 1;
    if (!four_step_tables(L, S, nhi, tw4_lo, tw4_hi))
        return false;
    hipStream_t s = default_stream();
    if (L == 65536 && prec == 4 && maxr >= 16 && pair_mode() != 0) {
        // single-pass tables, generated in FP64 and rounded once: W_L^(k1 m)
        // [32][2048], then W_2048^(m_lo q2) [128][16] and W_128^(m0 q1) [8][16]
        DevBuf t64;
        const size_t n4 = 32 * 2048, nb = 128 * 16 + 8 * 16;
        if (!t64.alloc((n4 + nb) * 16) || !pair_tw4.alloc(n4 * 8) || !pair_twb.alloc(nb * 8) ||
            !pair_err.alloc(256))
            return false;
        hipStream_t s = default_stream();
        char* b64 = (char*)t64.p;
        if (!hip_ok(launch_twiddle_2d(b64, 32, 2048, 65536, s), "pair tw4") ||
            !hip_ok(launch_twiddle_2d(b64 + n4 * 16, 128, 16, 2048, s), "pair twb1") ||
            !hip_ok(launch_twiddle_2d(b64 + (n4 + 128 * 16) * 16, 8, 16, 128, s), "pair twb2") ||
            !hip_ok(launch_convert_from_f64(4, pair_tw4.p, b64, n4, 1.0, s), "pair tw4 cvt") ||
            !hip_ok(launch_convert_from_f64(4, pair_twb.p, b64 + n4 * 16, nb, 1.0, s), "pair twb cvt") ||
            !hip_ok(launch_fill_u32((uint32_t*)pair_err.p, 64, 0u, s), "pair err") ||
            !hip_ok(hipStreamSynchronize(s), "pair tables"))
            return false;
        (void)num_cus(); // the XCD probe, here rather than inside an execution
        pair = true;
    }
    if (shaped_sub(N1, maxr) && shaped_sub(N2, maxr)) { // shaped passes use the default radices
        mixed_four = !fast_len_split(N1) || !fast_len_split(N2);
        // n entries of a table of this length and precision, generated in FP64 (gen)
        // and rounded once
        auto table = [&](SharedTab& t, uint32_t kind, uint64_t n, auto gen) -> bool {
            return t.get(kind + (prec == 8 ? 0u : 1u), L, 0, [&](DevBuf& d) {
                DevBuf f64;
                return f64.alloc(n * 16) && d.alloc(n * elem_bytes(prec)) &&
                       hip_ok(gen(f64.p), "four-step table") &&
                       hip_ok(launch_convert_from_f64(prec, d.p, f64.p, n, 1.0, s), "table cvt");
            });
        };
        if (!table(tw4_full, 10, L, [&](void* o) { return launch_twiddle_2d(o, N1, N2, L, s); }))
            return false;
        if (!mixed_four) {
            // the fused real-input rebuild's two factor tables
            const uint64_t ne = (uint64_t)N2 + 1;
            if (rebuilds &&
                (!table(rp_row, 12, N1,
                        [&](void* o) { return launch_twiddle_table(o, N1, 1, 2ull * L, s); }) ||
                 !table(rp_elem, 14, ne,
                        [&](void* o) { return launch_twiddle_table(o, ne, 1, 2ull * N2, s); })))
                return false;
            // and those of the inverse rebuild (without room for them: its own sweep)
            if (rebuilds && N1 >= 64 && N1 <= 1024 &&
                !inverse_rebuild_tables(L, N1, N2, prec, rq_row, rq_col))
                rq_row = rq_col = SharedTab();
            // a full table of 1 MiB or more falls out of the caches between the
            // pass-A tiles that share it, its two factors stay resident (measured:
            // the 2^16-point FP64 pass A fetched 139.7 MiB per 128 MiB group with
            // the full table, 128.3 with the factors)
            tw4_split = (uint64_t)L * elem_bytes(prec) >= (1u << 20);
            if (tw4_split && prec == 4) {
                auto rounded = [&](SharedTab& t, uint32_t kind, const SharedTab& from, uint64_t n) {
                    return t.get(kind, L, 0, [&](DevBuf& d) {
                        return d.alloc(n * 8) &&
                               hip_ok(launch_convert_from_f64(4, d.p, from.p, n, 1.0, s), "tw4 cvt");
                    });
                };
                if (!rounded(tw4s_hi, 20, tw4_hi, nhi) || !rounded(tw4s_lo, 21, tw4_lo, S))
                    return false;
            }
        }
    }
    return true;
}

// Tuning of the two-pass power-of-two path, fixed per process.
//  KFFT_AMD_CHUNK_MB: run the two passes over groups of transforms whose
//                     intermediate fits this many MiB, so the second pass can
//                     read part of it back from the caches (0: whole batch);
//                     with two streams a smaller batch of long transforms still
//                     runs as four groups
//  KFFT_AMD_NT:       non-temporal access bits: 1 pass-A input, 2 pass-B output,
//                     4 pass-A output, 8 pass-B input
//  KFFT_AMD_PIPE:     1: consecutive groups alternate between the caller's
//                     stream and a second library stream, so that one group's
//                     first pass runs beside the previous group's second pass
struct Tuning {
    // defaults measured on MI355X for 2^16 x 4096 (FP32 and FP64)
    size_t chunk_bytes = (size_t)128 << 20;
    uint32_t nt = 3;
    uint32_t pipe = 1;
};
static const Tuning& tuning() {
    static const Tuning t = [] {
        Tuning v;
        if (const char* c = getenv("KFFT_AMD_CHUNK_MB"))
            v.chunk_bytes = (size_t)(atof(c) * (1u << 20));
        if (const char* n = getenv("KFFT_AMD_NT"))
            v.nt = (uint32_t)atoi(n);
        if (const char* p = getenv("KFFT_AMD_PIPE"))
            v.pipe = (uint32_t)atoi(p);
        return v;
    }();
    return t;
}

// A second stream of the library (default priority), for work that runs beside
// the caller's stream within one execution; joined back before the execution
// returns.  It is created with a CU mask that names every CU: the runtime gives
// such a stream a hardware queue of its own, where an ordinary stream created
// after the process's queue limit (4 by default) shares one with an earlier
// stream, and two passes on one queue run one after the other (measured: the
// 2^16-point two-pass batch 1.54 ms instead of 1.41 in a process that had used
// both builds of the library).
static hipStream_t side_stream() {
    static std::once_flag once;
    static hipStream_t st = nullptr;
    std::call_once(once, [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            cus > 0) {
            std::vector<uint32_t> mask(((size_t)cus + 31) / 32, 0xffffffffu);
            if (cus % 32)
                mask.back() = (1u << (cus % 32)) - 1u;
            if (hipExtStreamCreateWithCUMask(&st, (uint32_t)mask.size(), mask.data()) == hipSuccess)
                return;
        }
        (void)hipGetLastError();
        if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) {
            (void)hipGetLastError();
            st = nullptr;
        }
    });
    return st;
}

// Work of one execution spread over the caller's stream s and the side stream:
// fork_side makes the side stream wait for what s holds so far (it returns the
// side stream, or nullptr when there is none: then everything stays on s), and
// join_side makes s wait for the side stream's work.
static hipStream_t fork_side(hipStream_t s, hipError_t* err) {
    *err = hipSuccess;
    hipStream_t s2 = side_stream();
    thread_local hipEvent_t ev = nullptr;
    if (s2 && !ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        ev = nullptr;
    }
    if (!s2 || !ev)
        return nullptr;
    hipError_t e = hipEventRecord(ev, s);
    if (e == hipSuccess)
        e = hipStreamWaitEvent(s2, ev, 0);
    *err = e;
    return e == hipSuccess ? s2 : nullptr;
}
static hipError_t join_side(hipStream_t s, hipStream_t s2) {
    if (!s2)
        return hipSuccess;
    thread_local hipEvent_t ev = nullptr;
    if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        ev = nullptr;
        return hipDeviceSynchronize(); // (no event: a full wait keeps the order)
    }
    hipError_t e = hipEventRecord(ev, s2);
    if (e == hipSuccess)
        e = hipStreamWaitEvent(s, ev, 0);
    return e;
}

// The fast passes fuse only conjugation (load / store) and scaling (store).
static bool fast_io_ok(const KfaIo& io, uint32_t allowed) {
    return (io.flags & ~allowed) == 0 && io.valid == 0xffffffffu && io.lo_mul == 0 &&
           io.e_mul == 1;
}

// a shaped pass of length L: the power-of-two passes, else the mixed-radix ones
static hipError_t launch_fast(int prec, uint32_t L, int mode, const FastArgs& a, hipStream_t s) {
    if (recorder())
        return hipErrorNotSupported; // shaped passes are not tasks of the ragged executor
    if ((L & (L - 1)) == 0)
        return prec == 8 ? launch_fast_f64(L, mode, a, s) : launch_fast_f32(L, mode, a, s);
    return prec == 8 ? launch_mixed_f64(L, mode, a, s) : launch_mixed_f32(L, mode, a, s);
}

// sub-lengths of the shaped two-pass forms: powers of two, and the mixed-radix
// sub-lengths where the plan keeps the default radix order (cap 16)
static bool shaped_sub(uint32_t N, uint32_t maxr) {
    return (fast_len_split(N) && maxr >= 16) || (mixed_sub_len(N) && maxr == 16);
}

// ============================================================== launch recorder
Recorder*& recorder() {
    thread_local Recorder* r = nullptr;
    return r;
}

hipError_t Recorder::add(uint32_t type, int prec, int maxe, uint32_t lds, uint64_t tiles,
                         uint32_t gx, const void* args, size_t bytes) {
    RecOp op;
    op.type = type;
    op.prec = (uint32_t)prec;
    op.maxe = (uint32_t)maxe;
    op.lds = lds;
    op.tiles = tiles;
    op.gx = gx;
    op.args.assign((const unsigned char*)args, (const unsigned char*)args + bytes);
    ops.push_back(std::move(op));
    return hipSuccess;
}

static FastArgs fast_args(const void* tw, uint64_t batch, double scale) {
    FastArgs f;
    memset(&f, 0, sizeof(f));
    f.tw = tw;
    f.batch = batch;
    f.scale = scale;
    f.in_C = f.out_C = 1;
    return f;
}

// Cooperative load/store order of a general pass: consecutive threads on
// consecutive instances when instances, not elements, are adjacent in memory
// (columns of a matrix, four-step passes), else along the elements.
static bool io_jfast(const KfaIo& io) {
    if (io.flags & KFA_IO_MAP)
        return false; // permuted elements: no order is coalesced
    const int64_t estep = (int64_t)io.e_mul * io.stride;
    if (estep == 1 || estep == -1)
        return false;
    int64_t istep;
    if (io.C > 1)
        istep = io.dist_lo + (int64_t)io.lo_mul * io.stride;
    else if (io.flags & KFA_IO_INST)
        return false; // instance bases come from a table
    else
        istep = io.dist_hi;
    return istep == 1 || istep == -1;
}

static uint32_t xcd_tile_order();

static hipError_t run_pass(const LdsPass& P, const KfaIo& in, const KfaIo& out, double scale,
                           double scale_post, uint64_t batch, const void* tw4_hi,
                           const void* tw4_lo, uint32_t tw4_n, uint32_t tw4_shift, hipStream_t s,
                           const void* mid_pw = nullptr, uint32_t mid_rows = 1,
                           void* mid_dc = nullptr, uint32_t dft = 0,
                           const void* dc_src = nullptr, bool dc_out = false) {
    KfaFftArgs a;
    memset(&a, 0, sizeof(a));
    a.mid_pw = (uint64_t)mid_pw;
    a.mid_dc = (uint64_t)mid_dc;
    a.mid_rows = mid_rows ? mid_rows : 1u;
    a.dc_src = (uint64_t)dc_src;
    a.dc_out = dc_out ? 1u : 0u;
    a.in = in;
    a.out = out;
    a.tw = (uint64_t)P.tw.p;
    a.tw4_hi = (uint64_t)tw4_hi;
    a.tw4_lo = (uint64_t)tw4_lo;
    a.tw4_n = tw4_n;
    a.tw4_shift = tw4_shift;
    a.scale = scale;
    a.scale_post = scale_post;
    a.batch = batch;
    a.L = P.L;
    a.nstages = P.nstages;
    a.tpi = P.tpi;
    a.in_jfast = io_jfast(in);
    a.out_jfast = io_jfast(out);
    a.ipw = P.pick_ipw(a.in_jfast || a.out_jfast);
    a.inst_stride = P.inst_stride;
    memcpy(a.st, P.st, sizeof(a.st));
    // FP64: stage twiddles in LDS when they fit beside the instances within what
    // keeps two workgroups per CU: each stage then reads them at LDS latency
    // instead of waiting on a memory round trip (the FP32 passes prefetch them)
    const size_t data = P.lds_bytes(a.ipw), twb = (size_t)P.tw_count * elem_bytes(P.prec);
    a.tw_lds = (P.prec == 8 && P.tw_count && data + twb <= 80 * 1024) ? P.tw_count : 0u;
    // XCD-contiguous tile order where the pass's instances are the columns or rows
    // of larger transforms (tiles of one transform then share an L2: measured 7%
    // faster on the 65536-point Rader convolution, 2% on 6561 = 81 x 81; one-pass
    // batches of whole transforms run 1-2% slower with it)
    // (rows in blocks of four columns share their lines with the next rows)
    const bool rows4 = ((in.flags | out.flags) & KFA_IO_BLK4) != 0;
    a.xcds = (!recorder() && (in.C > 1 || out.C > 1 || rows4)) ? xcd_tile_order() : 0u;
    // the shaped pass behind the same fused operations, where its length is
    // compiled and the radices are its schedule (not for split-operand stages,
    // not while recording tasks for the ragged executor)
    if (!recorder() && (P.prec == 8 || !dft)) {
        const hipError_t e = P.prec == 8 ? launch_mixgen_f64(a, s) : launch_mixgen_f32(a, s);
        if (e != hipErrorNotSupported)
            return e;
        (void)hipGetLastError();
    }
    if ((in.flags & KFA_IO_RPRE) || dc_out) // (callers ask Plan1D::fuses_real_pre, or
        return hipErrorNotSupported;        // store X[0] themselves)
    return launch_fft(P.prec, P.maxe, a, (uint32_t)(data + (a.tw_lds ? twb : 0)), s, dft);
}

// Both passes of the fast two-pass transform for `batch` contiguous instances.
hipError_t SubFft::run_four_fast(const KfaIo& load, const KfaIo& store, double scale,
                                 uint64_t batch, void* scratch, uint32_t nt,
                                 hipStream_t s, uint32_t dft) const {
    // pass A: columns n2 of length N1 (stride N2), W_L^(n2 k1) on store
    FastArgs a = fast_args(col.tw.p, batch * N2, 1.0);
    a.in = (const void*)load.ptr;
    a.in_C = N2;
    a.in_hi = load.dist_hi;
    a.in_lo = load.stride;
    a.in_stride = (int64_t)N2 * load.stride;
    a.out = scratch;
    a.out_C = N2;
    a.out_hi = L;
    a.out_lo = 1;
    a.out_stride = N2;
    a.tw4 = tw4_full.p;
    a.flags = KFA_FAST_TW4 | ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
              ((nt & 1) ? KFA_FAST_NT_IN : 0) | ((nt & 4) ? KFA_FAST_NT_OUT : 0) | dft;
    if (tw4_split) {
        a.flags |= KFA_FAST_TW4_SPLIT;
        a.tw4 = prec == 8 ? tw4_hi.p : tw4s_hi.p;
        a.tw4_lo = prec == 8 ? tw4_lo.p : tw4s_lo.p;
        a.tw4_shift = tw4_shift;
    }
    // FP64: XCD-contiguous tile order in both passes (measured: 2^20 x 16 and the
    // real 2^18 x 512 forward 14% faster, 2^16 x 4096 4%; the FP32 passes are
    // unchanged by it, and one-pass rows and 2D column passes slower)
    a.xcds = prec == 8 ? xcd_tile_order() : 0u;
    const bool rpre = (load.flags & KFA_IO_RPRE) != 0;
    if (rpre) { // bins are read twice: kept in the caches, on one XCD
        a.flags &= ~KFA_FAST_NT_IN;
        a.rpost_st = rq_row.p;
        a.rpost_w2 = rq_col.p;
        a.xcds = xcd_tile_order();
    }
    hipError_t e = launch_fast(prec, N1, rpre ? 3 : 1, a, s);
    if (e != hipSuccess)
        return e;
    // pass B: rows k1 of length N2, natural-order store X[k1 + N1 k2]
    FastArgs b = fast_args(row.tw.p, batch * N1, scale);
    b.in = scratch;
    b.in_C = N1;
    b.in_hi = L;
    b.in_lo = N2;
    b.in_stride = 1;
    b.out = (void*)store.ptr;
    b.out_C = N1;
    b.out_hi = store.dist_hi;
    b.out_lo = store.stride;
    b.out_stride = (int64_t)N1 * store.stride;
    b.flags = ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
              ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0) |
              ((nt & 2) ? KFA_FAST_NT_OUT : 0) | ((nt & 8) ? KFA_FAST_NT_IN : 0) | dft;
    if (store.flags & KFA_IO_RPOST) {
        // real-input rebuild in the store: X[0..L] of the 2L reals (no conjugation
        // or scaling reaches here)
        b.flags |= KFA_FAST_RPOST;
        b.rpost_st = rp_row.p;
        b.rpost_w2 = rp_elem.p;
    }
    b.xcds = a.xcds;
    return launch_fast(prec, N2, 2, b, s);
}

// Plain rows in one pass of the long-row form.
hipError_t SubFft::run_big(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                           hipStream_t s) const {
    KfaFftArgs a;
    memset(&a, 0, sizeof(a));
    a.in = load;
    a.out = store;
    a.tw = (uint64_t)big.tw.p;
    a.scale = scale;
    a.scale_post = 1.0;
    a.batch = batch;
    a.L = L;
    a.nstages = big.nstages;
    a.mid_rows = 1;
    return prec == 8 ? launch_bigrow_f64(a, s) : launch_bigrow_f32(a, s);
}

// Column four-step on row-major matrices: instance = column x of matrix m,
// element n at row n (pitch `stride`).  Pass A: for (n2, x), FFT over n1 of
// rows n1*N2 + n2, store k1 at row k1*N2 + n2 of the scratch (pitch C) times
// W_L^(n2 k1); pass B: for (k1, x), FFT over n2, store k2 at row k1 + N1*k2.
// One launch pair per matrix.
hipError_t SubFft::run_four_cols(const KfaIo& load, const KfaIo& store, double scale,
                                 uint64_t batch, void* scratch, uint32_t nt, hipStream_t s,
                                 uint32_t dft) const {
    const uint32_t X = load.C;
    const uint64_t nmat = batch / X;
    const int64_t esz = (int64_t)elem_bytes(prec);
    // matrices of 256 MiB and more run as four blocks of columns (multiples of
    // 64) whose pass pairs alternate between the caller's stream and the side
    // stream, so one block's first pass runs beside the previous block's
    // second.  The blocks of a stream share one part of the scratch, packed: its
    // lines are written again while the caches still hold them (measured, 8192^2
    // FP32 2D forward and inverse: one dispatch 1.37 ms, four blocks in columns of
    // the whole scratch 1.26-1.34, packed 1.21; eight packed blocks 1.25, sixteen
    // 1.28; blocks of the 69 MiB columns of the 4160^2 real convolution were 20%
    // slower than one dispatch each)
    const bool blocks = tuning().pipe && !no_alloc() && X >= 1024 &&
                        (size_t)L * X * (size_t)esz >= ((size_t)256 << 20);
    const uint32_t XB = blocks ? ((X / 4 + 63) / 64) * 64 : X;
    hipStream_t s2 = nullptr;
    if (XB < X) {
        hipError_t e;
        s2 = fork_side(s, &e);
        if (e != hipSuccess)
            return e;
    }
    for (uint64_t m = 0; m < nmat; ++m)
        for (uint32_t x0 = 0; x0 < X; x0 += XB) {
        // (a block keeps its stream and its part of the scratch in every matrix: each
        // part is then used in stream order)
        const uint32_t XC = std::min<uint32_t>(XB, X - x0);
        const hipStream_t sb = (s2 && ((x0 / XB) & 1)) ? s2 : s;
        FastArgs a = fast_args(col.tw.p, (uint64_t)N2 * XC, 1.0);
        a.in = (const void*)(load.ptr + (uint64_t)(((int64_t)m * load.dist_hi + x0) * esz));
        a.in_C = XC;
        a.in_hi = load.stride;
        a.in_lo = 1;
        a.in_stride = (int64_t)N2 * load.stride;
        char* sblk = (char*)scratch + ((x0 / XB) & 1) * (size_t)L * XB * esz;
        a.out = (void*)sblk;
        a.out_C = XC;
        a.out_hi = XB;
        a.out_lo = 1;
        a.out_stride = (int64_t)N2 * XB;
        a.tw4 = tw4_full.p;
        a.pad = N2;
        a.flags = KFA_FAST_TW4_HI | ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
                  ((nt & 1) ? KFA_FAST_NT_IN : 0) | dft;
        hipError_t e = launch_fast(prec, N1, 1, a, sb);
        if (e != hipSuccess)
            return e;
        FastArgs b = fast_args(row.tw.p, (uint64_t)N1 * XC, scale);
        b.in = (const void*)sblk;
        b.in_C = XC;
        b.in_hi = (int64_t)N2 * XB;
        b.in_lo = 1;
        b.in_stride = XB;
        b.out = (void*)(store.ptr + (uint64_t)(((int64_t)m * store.dist_hi + x0) * esz));
        b.out_C = XC;
        b.out_hi = store.stride;
        b.out_lo = 1;
        b.out_stride = (int64_t)N1 * store.stride;
        b.flags = ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
                  ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0) |
                  ((nt & 2) ? KFA_FAST_NT_OUT : 0) | dft;
        e = launch_fast(prec, N2, 1, b, sb);
        if (e != hipSuccess)
            return e;
    }
    return join_side(s, s2);
}

// Bluestein's convolution y = IDFT(DFT(x) * h) (unnormalised) with the load's
// element operations on x and the store's on y (whose CONJ1 finishes the
// inverse).  One LDS pass: both transforms in one workgroup tile, h applied in
// LDS between them.  Four-step L = N1 x N2 (C == 1 layouts): three passes over
// `scratch` (batch x L):
//   A1  columns n2: DFT over n1, times W_L^(n2 k1), into scratch[k1][n2]
//   M   rows k1 in place: DFT over n2 (spectrum index k1 + N1 k2), times
//       h[k1 + N1 k2] (hperm, laid out [k1][k2]), conjugate, DFT over k2 again,
//       times W_L^(k1 n2), conjugate: the row step of the inverse transform,
//       W_L^-(n2 + N2 n1)(k1 + N1 k2) = W_L^-(n2 k1) W_N2^-(n2 k2) W_N1^-(n1 k1)
//   A2  columns n2: conjugate, DFT over k1, store element n2 + N2 n1
// against four for two separate transforms.  `dc` (optional) receives the
// spectrum's element 0 per instance (Rader's A[0]).
hipError_t SubFft::run_conv(const KfaIo& load, const KfaIo& store, double scale,
                            double scale_post, uint64_t batch, const void* h, const void* hperm,
                            void* scratch, hipStream_t s, void* dc, uint32_t dft,
                            bool dc_out) const {
    if (three)
        return hipErrorNotSupported; // (Bluestein runs its steps separately there)
    if (!four)
        return run_pass(direct, load, store, scale, scale_post, batch, nullptr, nullptr, 0, 0, s, h,
                        1, dc_out ? nullptr : dc, dft, nullptr, dc_out);
    if (load.C != 1 || store.C != 1 || !hperm)
        return hipErrorInvalidValue;
    // A1: as pass A of the two-pass transform
    KfaIo ia = load;
    ia.C = N2;
    ia.dist_lo = 0;
    ia.lo_mul = 1;
    ia.e_mul = N2;
    ia.stride = load.stride;
    KfaIo oa;
    memset(&oa, 0, sizeof(oa));
    oa.ptr = (uint64_t)scratch;
    oa.C = N2;
    oa.dist_hi = L;
    oa.dist_lo = 1;
    oa.stride = N2;
    oa.e_mul = 1;
    oa.valid = 0xffffffffu;
    oa.flags = KFA_IO_TW4;
    hipError_t e = run_pass(col, ia, oa, 1.0, 1.0, batch * N2, tw4_hi.p, tw4_lo.p, L, tw4_shift, s,
                            nullptr, 1, nullptr, dft);
    if (e != hipSuccess)
        return e;
    // M: rows k1 of the scratch, in place
    KfaIo im;
    memset(&im, 0, sizeof(im));
    im.ptr = (uint64_t)scratch;
    im.C = N1;
    im.dist_hi = L;
    im.dist_lo = N2;
    im.stride = 1;
    im.e_mul = 1;
    im.valid = 0xffffffffu;
    KfaIo om = im;
    om.flags = KFA_IO_TW4 | KFA_IO_CONJ2;
    e = run_pass(row, im, om, 1.0, 1.0, batch * N1, tw4_hi.p, tw4_lo.p, L, tw4_shift, s, hperm, N1,
                 dc, dft);
    if (e != hipSuccess)
        return e;
    // A2: columns n2 of the scratch, conjugated, DFT over k1, stored at n2 + N2 n1
    KfaIo i2 = oa;
    i2.flags = KFA_IO_CONJ1;
    KfaIo o2 = store;
    o2.C = N2;
    o2.dist_lo = 0;
    o2.lo_mul = 1;
    o2.e_mul = N2;
    return run_pass(col, i2, o2, scale, scale_post, batch * N2, nullptr, nullptr, 0, 0, s, nullptr,
                    1, nullptr, dft, dc, dc_out);
}

// ============================================================ fused two-pass
static uint32_t env_u32(const char* name, uint32_t dflt) {
    const char* e = getenv(name);
    return e ? (uint32_t)atoi(e) : dflt;
}

static uint32_t g_num_cus = 0;

uint32_t num_cus() {
    xcd_queues();
    return g_num_cus;
}

uint32_t fused_queues() { return env_u32("KFFT_AMD_FUSED", 1) ? xcd_queues() : 0u; }

// XCD count when the probe saw workgroup b of an ordinary grid on XCD b mod n
// (round-robin dispatch), else 0 (atomic: plans may run on threads other than
// the one whose plan build ran the probe)
static std::atomic<uint32_t> g_xcd_rr{0};

uint32_t xcd_queues() {
    static std::once_flag once;
    static uint32_t nq = 0;
    std::call_once(once, [] {
        if (!runtime_init())
            return;
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            return;
        g_num_cus = (uint32_t)cus;
        const uint32_t groups = 2 * (uint32_t)cus;
        DevBuf ids;
        if (!ids.alloc(groups * 4))
            return;
        // nothing else of this process on the device while the probe runs: work
        // in flight on other streams holds CUs and changes where workgroups land
        hipStream_t s = default_stream();
        if (hipDeviceSynchronize() != hipSuccess ||
            launch_xcc_probe((uint32_t*)ids.p, groups, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return;
        std::vector<uint32_t> h(groups);
        if (hipMemcpy(h.data(), ids.p, groups * 4, hipMemcpyDeviceToHost) != hipSuccess)
            return;
        uint32_t seen = 0, maxid = 0;
        for (uint32_t v : h) {
            maxid = std::max(maxid, v);
            if (v < 32)
                seen |= 1u << v;
        }
        // every XCD from 0 to maxid must host workgroups of an ordinary grid
        if (maxid < 16 && seen == ((1u << (maxid + 1)) - 1) && maxid >= 1) {
            nq = maxid + 1;
            bool rr = true;
            for (uint32_t b = 0; b < groups; ++b)
                rr = rr && h[b] == b % nq;
            g_xcd_rr.store(rr ? nq : 0u, std::memory_order_relaxed);
        }
    });
    return nq;
}

// XCD-contiguous tile order of the general pass (KFFT_AMD_XCD_TILES=0 turns it
// off); 0 until a plan build has run the probe (no launch inside a transform)
static uint32_t xcd_tile_order() {
    static const bool on = [] {
        const char* e = getenv("KFFT_AMD_XCD_TILES");
        return !e || atoi(e) != 0;
    }();
    return on ? g_xcd_rr.load(std::memory_order_relaxed) : 0u;
}

hipError_t SubFft::run_fused(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                             hipStream_t s) const {
    std::lock_guard<std::mutex> lk(fused_mu);
    const uint32_t nq = fused_queues();
    const uint32_t S = env_u32("KFFT_AMD_FUSED_SLOTS", prec == 8 ? 4 : 6);
    const uint32_t wpc = env_u32("KFFT_AMD_FUSED_WGS", 2);
    const size_t words = 16 * (size_t)nq + 2 * batch + 1;
    if (!fused_ctr.ensure(words * 4) ||
        !fused_ring.ensure((size_t)nq * S * L * elem_bytes(prec)))
        return hipErrorOutOfMemory;
    hipError_t e = launch_fill_u32((uint32_t*)fused_ctr.p, words, 0u, s);
    if (e != hipSuccess)
        return e;
    FusedArgs f;
    memset(&f, 0, sizeof(f));
    f.in = (const void*)load.ptr;
    f.out = (void*)store.ptr;
    f.in_dist = load.dist_hi;
    f.out_dist = store.dist_hi;
    f.ring = fused_ring.p;
    f.tw_col = col.tw.p;
    f.tw_row = row.tw.p;
    f.tw4 = tw4_full.p;
    f.ctr = (uint32_t*)fused_ctr.p;
    f.T = batch;
    f.S = S;
    f.nq = nq;
    f.flags = ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
              ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
              ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0);
    f.spin_limit = 1u << 22;
    f.scale = scale;
    fused_T = batch;
    fused_used = true;
    const uint32_t groups = std::max<uint32_t>(nq, wpc * g_num_cus);
    return prec == 8 ? launch_fused_f64(N1, f, groups, s) : launch_fused_f32(N1, f, groups, s);
}

int SubFft::fused_error() const {
    std::lock_guard<std::mutex> lk(fused_mu);
    if (!fused_used || !fused_ctr.p)
        return 0;
    hipStream_t s = default_stream();
    uint32_t v = 0;
    const size_t off = (16 * (size_t)fused_queues() + 2 * fused_T) * 4;
    if (hipStreamSynchronize(s) != hipSuccess ||
        hipMemcpy(&v, (char*)fused_ctr.p + off, 4, hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    fused_used = false;
    return (int)v;
}

// ============================================================ single pass

// Pairs form at run time from the workgroups each XCD receives (XCC_ID), so
// the form needs only the XCD count, not any particular dispatch order.
uint32_t SubFft::pair_count(uint64_t batch) const {
    const uint32_t cus = num_cus(); // runs the XCD probe first if no plan build has
    const uint32_t X = xcd_queues();
    if (!pair || X < 1 || X > 16 || cus < 2 * X || batch == 0 || batch >= 0xffffffffull)
        return 0;
    uint32_t P = (cus / 2) / X * X;
    if (const char* e = getenv("KFFT_AMD_PAIRS")) {
        const uint32_t v = (uint32_t)atoi(e) / X * X;
        if (v >= X && v <= P)
            P = v;
    }
    const uint64_t want = (batch + X - 1) / X * X;
    return (uint32_t)std::min<uint64_t>(P, want);
}

// counter words of the single pass: a 1024-word header, then 160 per pair slot
static size_t pair_ctr_words(uint32_t P) { return 1024 + (size_t)160 * P; }

// inbox (2 P x 16384 values), then the counter words; 256-byte aligned parts
size_t SubFft::pair_scratch_bytes(uint64_t batch) const {
    const uint32_t P = pair_count(batch);
    if (!P)
        return 0;
    return (size_t)2 * P * 16384 * 8 + (pair_ctr_words(P) * 4 + 255) / 256 * 256;
}

hipError_t SubFft::run_pair(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                            void* scratch, hipStream_t s, uint32_t dft) const {
    const uint32_t P = pair_count(batch);
    if (!P || !scratch)
        return hipErrorInvalidValue;
    PairArgs a;
    memset(&a, 0, sizeof(a));
    a.in = (const void*)load.ptr;
    a.out = (void*)store.ptr;
    a.in_dist = load.dist_hi;
    a.out_dist = store.dist_hi;
    a.tw4 = pair_tw4.p;
    a.twb = pair_twb.p;
    a.inbox = scratch;
    a.ctr = (uint32_t*)((char*)scratch + (size_t)2 * P * 16384 * 8);
    a.err = (uint32_t*)pair_err.p;
    a.T = batch;
    a.npairs = P;
    a.nxcd = xcd_queues();
    a.spx = P / a.nxcd;
    a.flags = ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
              ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
              ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0);
    a.spin_limit = 1u << 23;
    a.scale = (float)scale;
    // pairs start in 16 groups 9000 cycles apart (measured: 2^16 x 4096 FP32
    // 2.06 ms without, 1.76 ms with; 8 groups 18000 apart 1.83 ms)
    a.stagger_groups = env_u32("KFFT_AMD_PAIR_GROUPS", 16);
    a.stagger_cycles = env_u32("KFFT_AMD_PAIR_CYCLES", 9000);
    hipError_t e = launch_fill_u32(a.ctr, pair_ctr_words(P), 0u, s);
    if (e != hipSuccess)
        return e;
    pair_used.store(true, std::memory_order_relaxed);
    return launch_pair_f32(a, dft, s);
}

int SubFft::pair_error() const {
    if (!pair || !pair_err.p || !pair_used.exchange(false, std::memory_order_relaxed))
        return 0;
    uint32_t v = 0;
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(&v, pair_err.p, 4, hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    if (v) {
        const uint32_t z = 0;
        (void)hipMemcpy(pair_err.p, &z, 4, hipMemcpyHostToDevice);
    }
    return (int)v;
}

size_t SubFft::scratch_elems(uint64_t batch) const {
    if (three) // one transform's column pass output, then the inner plan's scratch
        return (size_t)L + 256 + inner->scratch_bytes(N1) / elem_bytes(prec);
    const size_t two = four ? (size_t)batch * L : 0;
    const size_t one = pair ? (pair_scratch_bytes(batch) + 2 * (size_t)prec - 1) / (2 * prec) : 0;
    return two > one ? two : one;
}

// Per transform: pass A = columns n2 of length N1 (stride N2) into the scratch,
// times W_L^(n2 k1) (conjugated there when the store conjugates, so that the
// inner plan's inverse, conj(DFT(conj(.))), completes conj(DFT(.))); then the
// inner plan over the N1 rows of N2, storing X[k1 + N1 k2].
hipError_t SubFft::run_three(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                             void* scratch, hipStream_t s, uint32_t dft) const {
    if (!fast_io_ok(load, KFA_IO_CONJ1) || !fast_io_ok(store, KFA_IO_CONJ2 | KFA_IO_SCALE) ||
        load.C != 1 || store.C != 1 || recorder())
        return hipErrorInvalidValue;
    const int64_t esz = (int64_t)elem_bytes(prec);
    char* sa = (char*)scratch;
    char* sb = sa + ((size_t)L * esz + 255) / 256 * 256;
    const bool inv = (store.flags & KFA_IO_CONJ2) != 0;
    const double sc = (store.flags & KFA_IO_SCALE) ? scale : 1.0;
    for (uint64_t t = 0; t < batch; ++t) {
        KfaIo ia = load;
        ia.ptr = load.ptr + (uint64_t)((int64_t)t * load.dist_hi * esz);
        ia.dist_hi = 0;
        ia.C = N2;
        ia.dist_lo = 0;
        ia.lo_mul = 1;
        ia.e_mul = N2;
        KfaIo oa;
        memset(&oa, 0, sizeof(oa));
        oa.ptr = (uint64_t)sa;
        oa.C = N2;
        oa.dist_lo = 1;
        oa.stride = N2;
        oa.e_mul = 1;
        oa.valid = 0xffffffffu;
        oa.flags = KFA_IO_TW4 | (inv ? KFA_IO_CONJ2 : 0);
        hipError_t e = run_pass(col, ia, oa, 1.0, 1.0, N2, tw4_hi.p, tw4_lo.p, L, tw4_shift, s,
                                nullptr, 1, nullptr, dft);
        if (e != hipSuccess)
            return e;
        Layout li, lo;
        li.ptr = sa;
        li.dist_hi = N2;
        lo.ptr = (void*)(store.ptr + (uint64_t)((int64_t)t * store.dist_hi * esz));
        lo.dist_hi = store.stride;
        lo.stride = (int64_t)N1 * store.stride;
        e = inner->execute(li, lo, N1, inv, sc, sb, s);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

bool SubFft::rpost_two_pass() const {
    if (!four || !tw4_full.p || !rp_row.p || N2 < 32 || N1 < 2)
        return false;
    const uint32_t ipw = prec == 8 ? fast_tout_ipw_f64(N2) : fast_tout_ipw_f32(N2);
    return ipw >= 2 && ipw % 2 == 0 && N1 % ipw == 0;
}

// KFFT_AMD_TRACE=1: one line on stderr per two-pass-length execution naming
// the form it takes (read at every call, so a process can switch it on late)
static bool trace_on() {
    const char* e = getenv("KFFT_AMD_TRACE");
    return e && e[0] == '1';
}
static void trace_path(uint32_t L, int prec, uint64_t batch, const char* form) {
    if (trace_on())
        fprintf(stderr, "kfft_amd: %u-point %s x %llu: %s\n", L, prec == 8 ? "FP64" : "FP32",
                (unsigned long long)batch, form);
}

hipError_t SubFft::run(const KfaIo& load, const KfaIo& store, double scale, double scale_post,
                       uint64_t batch, void* scratch, hipStream_t s, bool onchip,
                       uint32_t dft) const {
    const bool simple = fast_io_ok(load, KFA_IO_CONJ1) &&
                        fast_io_ok(store, KFA_IO_CONJ2 | KFA_IO_SCALE) && scale_post == 1.0;
    const bool rec = recorder() != nullptr; // recording for the ragged executor: general passes
    if (three) {
        if (scale_post != 1.0 || !simple)
            return hipErrorInvalidValue;
        trace_path(L, prec, batch, "three passes");
        return run_three(load, store, scale, batch, scratch, s, dft);
    }
    // both shaped passes over groups of transforms whose intermediate fits the
    // chunk size (the second pass then reads part of it back from the caches)
    auto four_fast_chunked = [&]() -> hipError_t {
        const Tuning& tn = tuning();
        uint64_t chunk = batch;
        if (tn.chunk_bytes) {
            chunk = tn.chunk_bytes / ((size_t)L * elem_bytes(prec));
            // long transforms (fewer than 64 per group): a batch of fewer than
            // four groups runs as four, so that the two streams overlap
            // (measured: 2^20 x 16 FP64 in four groups of 64 MiB 0.278 ms against
            // 0.304 in two of 128 MiB; 6561 x 2560 unchanged either way)
            if (tn.pipe && chunk < 64 && batch < 4 * chunk && batch >= 4)
                chunk = (batch + 3) / 4;
            chunk = std::max<uint64_t>(1, std::min<uint64_t>(chunk, batch));
        }
        const int64_t esz = (int64_t)elem_bytes(prec);
        // two groups in flight: group c runs on stream c mod 2 with its own half
        // of the scratch (the scratch holds the whole batch, so two groups fit)
        const bool two = tn.pipe && batch >= 2 * chunk && !no_alloc();
        hipStream_t s2 = nullptr;
        if (two) {
            hipError_t e;
            s2 = fork_side(s, &e);
            if (e != hipSuccess)
                return e;
        }
        const size_t chunk_bytes = (size_t)chunk * L * elem_bytes(prec);
        uint64_t c = 0;
        for (uint64_t c0 = 0; c0 < batch; c0 += chunk, ++c) {
            const uint64_t nb = std::min<uint64_t>(chunk, batch - c0);
            KfaIo ld = load, st = store;
            ld.ptr += (uint64_t)((int64_t)c0 * load.dist_hi * esz);
            st.ptr += (uint64_t)((int64_t)c0 * store.dist_hi * esz);
            const bool odd = s2 && (c & 1);
            void* sc = odd ? (void*)((char*)scratch + chunk_bytes) : scratch;
            hipError_t e = run_four_fast(ld, st, scale, nb, sc, tn.nt, odd ? s2 : s, dft);
            if (e != hipSuccess)
                return e;
        }
        return join_side(s, s2);
    };
    if (four && (store.flags & KFA_IO_RPOST)) {
        // fused rebuild: the shaped two-pass form on plain contiguous rows only
        KfaIo st = store;
        st.flags &= ~KFA_IO_RPOST;
        if (rec || !rpost_two_pass() || load.C != 1 || store.C != 1 || scale_post != 1.0 ||
            !fast_io_ok(load, 0) || !fast_io_ok(st, 0))
            return hipErrorInvalidValue;
        // whole batch: groups on two streams measured slower here (2^18 x 512 in 2, 4
        // or 8 groups: 1.06-1.07 against 1.03 ms)
        return run_four_fast(load, store, scale, batch, scratch, tuning().nt, s, dft);
    }
    // (in place or on buffers apart: a workgroup stores its row over no other that is
    // still to be read, as the two passes do through their scratch)
    auto rows_safe = [&] {
        const int64_t esz = (int64_t)elem_bytes(prec);
        if (load.ptr == store.ptr && load.dist_hi == store.dist_hi)
            return true;
        const uint64_t ispan = ((batch - 1) * (uint64_t)load.dist_hi + L) * esz;
        const uint64_t ospan = ((batch - 1) * (uint64_t)store.dist_hi + L) * esz;
        return load.dist_hi >= 0 && store.dist_hi >= 0 &&
               (load.ptr + ispan <= store.ptr || store.ptr + ospan <= load.ptr);
    };
    if (big.L && simple && !rec && !dft && load.C == 1 && store.C == 1 && load.stride == 1 &&
        store.stride == 1 && !onchip && batch >= num_cus() && batch <= 0x7fffffffull &&
        rows_safe())
        // (a row per CU at least: 100 rows of 6561 take 21.7 us here, 18.7 in the two
        // passes, whose tiles split a row over several workgroups)
        return run_big(load, store, scale, batch, s);
    if (four && (load.flags & KFA_IO_RPRE)) {
        // inverse rebuild in pass A's load: as above
        KfaIo ld = load;
        ld.flags &= ~KFA_IO_RPRE;
        if (rec || !rq_row.p || dft || load.C != 1 || store.C != 1 || scale_post != 1.0 ||
            load.stride != 1 || !fast_io_ok(ld, KFA_IO_CONJ1) ||
            !fast_io_ok(store, KFA_IO_CONJ2 | KFA_IO_SCALE))
            return hipErrorInvalidValue;
        return four_fast_chunked();
    }
    if (!four) {
        if (simple && fast_len(L) && !rec && maxr >= 16) {
            const bool rows = load.C == 1 && store.C == 1 && load.stride == 1 && store.stride == 1;
            const bool cols = load.C == store.C && load.dist_lo == 1 && store.dist_lo == 1 &&
                              load.stride != 1 && store.stride != 1 && fast_len_split(L);
            if (rows || cols) {
                FastArgs f = fast_args(direct.tw.p, batch, scale);
                f.in = (const void*)load.ptr;
                f.out = (void*)store.ptr;
                f.in_C = load.C;
                f.in_hi = load.dist_hi;
                f.in_lo = load.dist_lo;
                f.in_stride = load.stride;
                f.out_C = store.C;
                f.out_hi = store.dist_hi;
                f.out_lo = store.dist_lo;
                f.out_stride = store.stride;
                f.flags = ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
                          ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
                          ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0) | dft;
                return launch_fast(prec, L, rows ? 0 : 1, f, s);
            }
        }
        // mixed-radix lengths: the shaped row pass where it is compiled (its radix
        // order is radix_list's at the default cap, so it shares direct.tw)
        if (simple && mixed_len(L) && !rec && maxr == 16 && !dft && load.C == 1 &&
            store.C == 1 && load.stride == 1 && store.stride == 1) {
            FastArgs f = fast_args(direct.tw.p, batch, scale);
            f.in = (const void*)load.ptr;
            f.out = (void*)store.ptr;
            f.in_C = 1;
            f.in_hi = load.dist_hi;
            f.in_stride = 1;
            f.out_C = 1;
            f.out_hi = store.dist_hi;
            f.out_stride = 1;
            f.flags = ((load.flags & KFA_IO_CONJ1) ? KFA_FAST_CONJ_IN : 0) |
                      ((store.flags & KFA_IO_CONJ2) ? KFA_FAST_CONJ_OUT : 0) |
                      ((store.flags & KFA_IO_SCALE) ? KFA_FAST_SCALE : 0);
            const hipError_t e = prec == 8 ? launch_mixed_f64(L, 0, f, s) : launch_mixed_f32(L, 0, f, s);
            if (e != hipErrorNotSupported)
                return e;
            (void)hipGetLastError();
        }
        return run_pass(direct, load, store, scale, scale_post, batch, nullptr, nullptr, 0, 0, s,
                        nullptr, 1, nullptr, dft);
    }
    // (the mixed-radix shaped passes have no split-operand form)
    const bool shaped4 = tw4_full.p && !(dft && mixed_four && prec == 4);
    if (simple && shaped4 && !rec && load.C > 1 && store.C == load.C && load.dist_lo == 1 &&
        store.dist_lo == 1 && load.stride > 0 && store.stride > 0 && batch % load.C == 0)
        return run_four_cols(load, store, scale, batch, scratch, tuning().nt, s, dft);
    if (load.C != 1 || store.C != 1)
        return hipErrorInvalidValue;
    // on-chip forms: the single pass by workgroup pairs (FP32), else the fused
    // persistent two-pass kernel (FP64)
    if (onchip && trace_on())
        fprintf(stderr, "kfft_amd: on-chip request: pair tables %d, XCD order %u, CUs %u, "
                        "plain io %d, recording %d, no-alloc %d\n",
                (int)pair, xcd_tile_order(), num_cus(), (int)simple, (int)rec, (int)no_alloc());
    if (pair && (onchip || pair_mode() == 1) && simple && !rec && load.stride == 1 &&
        store.stride == 1 && pair_count(batch)) {
        trace_path(L, prec, batch, "single pass by workgroup pairs");
        return run_pair(load, store, scale, batch, scratch, s, dft);
    }
    if (onchip && !pair && !rec && !dft && !no_alloc() && simple && tw4_full.p && N1 == 256 && N2 == 256 &&
        s == default_stream() && load.stride == 1 && store.stride == 1 && fused_queues() > 0) {
        trace_path(L, prec, batch, "fused two-pass kernel");
        return run_fused(load, store, scale, batch, s);
    }
    if (simple && shaped4 && !rec) {
        trace_path(L, prec, batch, "two shaped passes");
        return four_fast_chunked();
    }
    trace_path(L, prec, batch, "two general passes");
    // pass A: columns of length N1 (stride N2), twiddle W_L^(n2 k1) on store
    KfaIo ia = load;
    ia.C = N2;
    ia.dist_lo = 0;
    ia.lo_mul = 1;
    ia.e_mul = N2;
    ia.stride = load.stride;
    KfaIo oa;
    memset(&oa, 0, sizeof(oa));
    oa.ptr = (uint64_t)scratch;
    oa.C = N2;
    oa.dist_hi = L;
    oa.dist_lo = 1;
    oa.stride = N2;
    oa.lo_mul = 0;
    oa.e_mul = 1;
    oa.valid = 0xffffffffu;
    oa.flags = KFA_IO_TW4;
    hipError_t e = run_pass(col, ia, oa, 1.0, scale_post, batch * N2, tw4_hi.p, tw4_lo.p, L,
                            tw4_shift, s, nullptr, 1, nullptr, dft);
    if (e != hipSuccess)
        return e;
    // pass B: rows of length N2, transposed store X[k1 + N1 k2]
    KfaIo ib;
    memset(&ib, 0, sizeof(ib));
    ib.ptr = (uint64_t)scratch;
    ib.C = N1;
    ib.dist_hi = L;
    ib.dist_lo = N2;
    ib.stride = 1;
    ib.lo_mul = 0;
    ib.e_mul = 1;
    ib.valid = 0xffffffffu;
    KfaIo ob = store;
    ob.C = N1;
    ob.dist_lo = 0;
    ob.aux_dist_lo = 0;
    ob.lo_mul = 1;
    ob.e_mul = N1;
    return run_pass(row, ib, ob, scale, scale_post, batch * N1, nullptr, nullptr, 0, 0, s, nullptr,
                    1, nullptr, dft);
}

// ==================================================================== Plan1D
static bool is_prime(uint32_t n) {
    if (n < 2)
        return false;
    for (uint64_t d = 2; d * d <= n; ++d)
        if (n % d == 0)
            return false;
    return true;
}

static uint64_t powmod(uint64_t b, uint64_t e, uint64_t m) {
    uint64_t r = 1 % m;
    b %= m;
    while (e) {
        if (e & 1)
            r = r * b % m;
        b = b * b % m;
        e >>= 1;
    }
    return r;
}

static uint32_t primitive_root(uint32_t p) {
    std::vector<uint32_t> f;
    uint32_t m = p - 1;
    for (uint32_t d = 2; (uint64_t)d * d <= m; ++d)
        if (m % d == 0) {
            f.push_back(d);
            while (m % d == 0)
                m /= d;
        }
    if (m > 1)
        f.push_back(m);
    for (uint32_t g = 2; g < p; ++g) {
        bool ok = true;
        for (uint32_t q : f)
            if (powmod(g, (p - 1) / q, p) == 1) {
                ok = false;
                break;
            }
        if (ok)
            return g;
    }
    return 0;
}

static KfaIo io_plain(void* ptr, int64_t dist_hi) {
    KfaIo io;
    memset(&io, 0, sizeof(io));
    io.ptr = (uint64_t)ptr;
    io.C = 1;
    io.dist_hi = dist_hi;
    io.stride = 1;
    io.e_mul = 1;
    io.valid = 0xffffffffu;
    return io;
}

static KfaIo io_from(const Layout& l) {
    KfaIo io;
    memset(&io, 0, sizeof(io));
    io.ptr = (uint64_t)l.ptr;
    io.C = l.C ? l.C : 1;
    io.dist_hi = l.dist_hi;
    io.dist_lo = l.dist_lo;
    io.stride = l.stride;
    io.e_mul = 1;
    io.valid = 0xffffffffu;
    io.flags = l.flags & (KFA_IO_REAL | KFA_IO_REAL_PAIRS | KFA_IO_BLK4);
    if (l.inst) {
        io.inst = (uint64_t)l.inst;
        io.flags |= KFA_IO_INST;
    }
    if (l.real_pre) {
        io.pw = (uint64_t)l.real_pre;
        io.flags |= KFA_IO_RPRE;
    }
    if (l.real_post) {
        io.pw = (uint64_t)l.real_post;
        io.flags |= KFA_IO_RPOST;
    }
    return io;
}

// FFT of a double-precision table with a temporary double-precision plan,
// then rounded once into the plan precision.
static bool fft_table_f64(uint32_t L, const void* src64, DevBuf& dst, int prec, double scale) {
    SubFft f;
    f.rebuilds = false;
    if (!f.plan(L, 8))
        return false;
    DevBuf out64, scr;
    if (!out64.alloc((size_t)L * 16) || !scr.alloc(std::max<size_t>(16, f.scratch_elems(1) * 16)))
        return false;
    hipStream_t s = default_stream();
    KfaIo in = io_plain((void*)src64, L), out = io_plain(out64.p, L);
    if (!hip_ok(f.run(in, out, 1.0, 1.0, 1, scr.p, s), "table fft"))
        return false;
    if (!dst.alloc((size_t)L * elem_bytes(prec)))
        return false;
    if (!hip_ok(launch_convert_from_f64(prec, dst.p, out64.p, L, scale, s), "convert"))
        return false;
    return hip_ok(hipStreamSynchronize(s), "table sync");
}

// the smallest 2,3,5-smooth length from n on with a plan (0: none)
static uint32_t smooth_at_least(uint64_t n, int prec) {
    for (uint64_t m = n; m < (1ull << 32); ++m) {
        uint64_t r = m;
        for (uint64_t p : {2ull, 3ull, 5ull})
            while (r % p == 0)
                r /= p;
        if (r == 1 && subfft_capable((uint32_t)m, prec))
            return (uint32_t)m;
    }
    return 0;
}

uint32_t blue_length(uint32_t n, int prec, bool pow2) {
    const uint64_t need = 2ull * n - 1;
    if (pow2) {
        uint64_t m = 1;
        while (m < need)
            m <<= 1;
        if (m < (1ull << 32) && subfft_capable((uint32_t)m, prec))
            return (uint32_t)m;
    }
    return smooth_at_least(need, prec);
}

// Bluestein with a power-of-two convolution length wherever its passes are the
// shaped ones compiled for it (one pass, or two factors of 64 to 1024): up to
// twice the points of the smooth length, in passes several times as fast as the
// general ones.  Not where only the smooth length fits one pass, nor where only
// it leaves enough columns per workgroup for column layouts.  Measured, smooth ->
// power of two: one 94132-point call FP64 80 -> 49 us, 94132 x 64 FP64 675 -> 354,
// 1069 x 8000 FP64 380 -> 238, 4415 x 4000 FP32 1225 -> 663, 74 x 100000 FP32 189 -> 65;
// with the most points for it (1.9 times) 33331 x 300 FP64 1287 -> 705, 2134 x 2000 FP64
// 318 -> 251, 66191 x 63 FP64 440 -> 327, 264765 x 15 FP64 462 -> 360.
PlanVariant default_variant(uint32_t n, int prec) {
    PlanVariant v;
    if (n < 2 || subfft_capable(n, prec) || (is_prime(n) && subfft_capable(n - 1, prec, false)))
        return v;
    const uint64_t need = 2ull * n - 1;
    uint64_t p2 = 1;
    while (p2 < need)
        p2 <<= 1;
    if (p2 > (1u << 20))
        return v;
    const uint32_t m = blue_length(n, prec, false);
    const bool one2 = p2 <= direct_max(prec);
    const bool one = m <= direct_max(prec) || mixed_len(m);
    const uint64_t cols = 72 * 1024 / (8 * elem_bytes(prec)) * 16 / 17; // LdsPass::pick_ipw
    v.pow2_m = (one2 || !one) && !(m <= cols && p2 > cols);
    return v;
}

// For a four-step inner transform, the convolution's middle pass reads the
// spectrum table h in its row order: out[k1 * N2 + k2] = h[k1 + N1 k2].
static bool conv_table_rows(const DevBuf& h, const SubFft& sub, DevBuf& out) {
    if (!sub.four)
        return true;
    const size_t eb = elem_bytes(sub.prec);
    hipStream_t s = default_stream();
    return out.alloc((size_t)sub.L * eb) &&
           hip_ok(launch_transpose((int)eb, h.p, out.p, sub.N1, sub.N2, 1, s), "conv table rows") &&
           hip_ok(hipStreamSynchronize(s), "conv table rows");
}

bool Plan1D::build() {
    if (!runtime_init())
        return false;
    xcd_queues(); // the dispatch-order probe, once per process
    if (n_ == 0) {
        set_error("zero length");
        return false;
    }
    hipStream_t s = default_stream();
    if (n_ == 1 || subfft_capable(n_, prec_)) {
        kind_ = n_ == 1 ? Kind::Identity : Kind::Direct;
        if (n_ == 1) {
            sub_.L = 1;
            sub_.prec = prec_;
            sub_.four = false;
            return sub_.direct.plan(1, prec_);
        }
        return sub_.plan(n_, prec_, var_.four, var_.maxr);
    }
    // (Rader's convolution runs on a one- or two-pass inner transform)
    if (is_prime(n_) && subfft_capable(n_ - 1, prec_, false)) {
        kind_ = Kind::Rader;
        const uint32_t L = n_ - 1, g = primitive_root(n_);
        const uint32_t ginv = (uint32_t)powmod(g, n_ - 2, n_);
        std::vector<uint32_t> q(L), p(L);
        uint64_t a = 1, b = 1;
        for (uint32_t k = 0; k < L; ++k) {
            q[k] = (uint32_t)a;
            p[k] = (uint32_t)b;
            a = a * g % n_;
            b = b * ginv % n_;
        }
        if (!qidx_.alloc(L * 4) || !pidx_.alloc(L * 4))
            return false;
        if (!hip_ok(hipMemcpy(qidx_.p, q.data(), L * 4, hipMemcpyHostToDevice), "qidx") ||
            !hip_ok(hipMemcpy(pidx_.p, p.data(), L * 4, hipMemcpyHostToDevice), "pidx"))
            return false;
        DevBuf b64;
        if (!b64.alloc((size_t)L * 16))
            return false;
        if (!hip_ok(launch_twiddle_indexed(b64.p, (const uint32_t*)pidx_.p, L, n_, 0, s), "rader b"))
            return false;
        if (!fft_table_f64(L, b64.p, bhat_, prec_, 1.0))
            return false;
        sub_.rebuilds = false;
        if (!sub_.plan(L, prec_, var_.four, var_.maxr))
            return false;
        return conv_table_rows(bhat_, sub_, hperm_);
    }
    kind_ = Kind::Bluestein;
    M_ = blue_length(n_, prec_, var_.pow2_m);
    if (!M_) {
        set_error("no Bluestein length for " + std::to_string(n_));
        return false;
    }
    DevBuf c64, h64;
    if (!c64.alloc((size_t)n_ * 16) || !h64.alloc((size_t)M_ * 16))
        return false;
    if (!hip_ok(launch_bluestein_tables(c64.p, h64.p, n_, M_, s), "bluestein tables"))
        return false;
    if (!fft_table_f64(M_, h64.p, hhat_, prec_, 1.0))
        return false;
    if (!chirp_.alloc((size_t)n_ * elem_bytes(prec_)))
        return false;
    if (!hip_ok(launch_convert_from_f64(prec_, chirp_.p, c64.p, n_, 1.0, s), "chirp"))
        return false;
    if (!hip_ok(hipStreamSynchronize(s), "bluestein sync"))
        return false;
    sub_.rebuilds = false;
    if (!sub_.plan(M_, prec_, var_.four, var_.maxr))
        return false;
    return conv_table_rows(hhat_, sub_, hperm_);
}

void cost_features(uint32_t n, uint32_t kind, uint32_t count, int prec, const RaggedChoice& c,
                   float* f) {
    const bool half = kind == RAGGED_REAL && n % 2 == 0;
    const uint32_t plen = half ? n / 2 : n;
    uint32_t L = plen;
    float rader = 0.0f, blue = 0.0f;
    if (plen > 1 && !subfft_capable(plen, prec, false)) {
        if (is_prime(plen) && subfft_capable(plen - 1, prec, false)) {
            rader = 1.0f;
            L = plen - 1;
        } else {
            blue = 1.0f;
            L = blue_length(plen, prec, c.v.pow2_m);
        }
    }
    int e[6] = {0, 0, 0, 0, 0, 0};
    uint32_t m = std::max<uint32_t>(L, 1);
    const uint32_t primes[] = {2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31};
    const int slot[] = {0, 1, 2, 3, 4, 4, 5, 5, 5, 5, 5};
    for (int i = 0; i < 11; ++i)
        while (m % primes[i] == 0) {
            m /= primes[i];
            ++e[slot[i]];
        }
    const float scale[6] = {17.0f, 11.0f, 7.0f, 6.0f, 5.0f, 4.0f};
    for (int i = 0; i < 6; ++i)
        f[i] = (float)e[i] / scale[i];
    f[6] = rader;
    f[7] = blue;
    f[8] = (float)std::log2((double)std::max<uint32_t>(n, 1)) / 16.0f;
    f[9] = (float)std::log2((double)std::max<uint32_t>(L, 1)) / 18.0f;
    f[10] = (float)std::log2((double)std::max<uint32_t>(count, 1)) / 14.0f;
    f[11] = kind == RAGGED_REAL ? 1.0f : 0.0f;
    f[12] = prec == 8 ? 1.0f : 0.0f;
    f[13] = c.v.maxr >= 16 ? 1.0f : 0.0f;
    f[14] = (c.v.maxr >= 8 && c.v.maxr < 16) ? 1.0f : 0.0f;
    f[15] = c.v.maxr < 8 ? 1.0f : 0.0f;
    f[16] = c.v.four ? 1.0f : 0.0f;
    f[17] = c.ipw_cap ? (float)std::log2((double)c.ipw_cap) / 8.0f : 1.0f;
    f[18] = (!c.v.four && L > 1 && lds_capable(L, prec) &&
             (L <= direct_max(prec) || !split_four(L, prec, &m, &m)))
                ? 1.0f
                : 0.0f;
}

bool choice_applies(uint32_t n, uint32_t kind, int prec, const RaggedChoice& c) {
    const uint32_t plen = (kind == RAGGED_REAL && n % 2 == 0) ? n / 2 : n;
    const bool blue = plen > 1 && !subfft_capable(plen, prec, false) &&
                      !(is_prime(plen) && subfft_capable(plen - 1, prec, false));
    if (c.v.pow2_m && !blue)
        return false; // the power-of-two convolution length is a Bluestein choice
    if (!c.v.four)
        return true;
    uint32_t L = plen, a, b;
    if (plen > 1 && !subfft_capable(plen, prec, false))
        L = blue ? blue_length(plen, prec, c.v.pow2_m) : plen - 1;
    return L > 1 && split_four(L, prec, &a, &b);
}

std::vector<RaggedChoice> tune_candidates() {
    std::vector<RaggedChoice> v;
    for (uint32_t maxr : {16u, 8u, 4u})
        for (bool four : {false, true})
            for (uint32_t cap : {0u, 16u, 4u, 1u}) {
                RaggedChoice c;
                c.v.maxr = maxr;
                c.v.four = four;
                c.ipw_cap = cap;
                v.push_back(c);
            }
    // Bluestein classes: a power-of-two convolution length, whose passes run
    // as the executor's compiled shaped tiles, against the shortest smooth one
    for (bool four : {false, true}) {
        RaggedChoice c;
        c.v.pow2_m = true;
        c.v.four = four;
        v.push_back(c);
    }
    return v;
}

const char* Plan1D::describe(bool onchip) const {
    char buf[256];
    const char* k = kind_ == Kind::Identity ? "identity"
                    : kind_ == Kind::Direct ? "direct"
                    : kind_ == Kind::Rader  ? "rader"
                                            : "bluestein";
    if (sub_.three)
        snprintf(buf, sizeof buf, "%s n=%u inner=%u three-pass %u x %u", k, n_, sub_.L, sub_.N1,
                 sub_.N2);
    else if (sub_.four)
        snprintf(buf, sizeof buf, "%s n=%u inner=%u four-step %ux%u", k, n_, sub_.L, sub_.N1,
                 sub_.N2);
    else
        snprintf(buf, sizeof buf, "%s n=%u inner=%u one-pass", k, n_, sub_.L);
    desc_ = buf;
    if (var_.maxr < 16)
        desc_ += " maxradix=" + std::to_string(var_.maxr);
    if (kind_ == Kind::Direct && !sub_.four && var_.maxr == 16 && mixed_len(sub_.L))
        desc_ += ", shaped mixed-radix rows";
    if (kind_ == Kind::Direct && sub_.big.L)
        desc_ += ", large batches of rows in one pass";
    if (onchip && sub_.pair)
        desc_ += ", on-chip form: single pass 32x2048 by workgroup pairs";
    return desc_.c_str();
}

bool Plan1D::supports_columns() const {
    // one-pass plans whose column tiles hold enough columns (>= 8) for coalesced
    // rows of memory; longer columns are better served by tiled transposes
    return !sub_.four && !sub_.three && sub_.direct.pick_ipw(true) >= 8;
}

bool Plan1D::supports_plain_columns() const {
    // as supports_columns, plus Direct four-step plans on the shaped passes (column
    // four-step), whose mixed-radix halves have no split-operand form (FP32)
    const bool shaped4 = sub_.tw4_full.p && !(sub_.mixed_four && prec_ == 4 && split_dft_default());
    return supports_columns() || (kind_ == Kind::Direct && sub_.four && shaped4);
}

size_t Plan1D::scratch_bytes(uint64_t batch) const {
    const size_t eb = elem_bytes(prec_);
    size_t elems = sub_.scratch_elems(batch);
    if (kind_ == Kind::Rader) // x0, A[0] (each 256-byte aligned), the convolution's scratch
        return (2 * ((batch * eb + 255) / 256) * 256) + (size_t)batch * sub_.L * eb + 256;
    if (kind_ == Kind::Bluestein) // the convolution's four-step scratch, or for a
        // three-pass inner length one zero-padded transform and its passes' scratch
        elems = sub_.three  ? (size_t)sub_.L + 256 + sub_.scratch_elems(1)
                : sub_.four ? (size_t)batch * sub_.L
                            : 0;
    return elems * eb + 256;
}

size_t Plan1D::scratch_charge(uint64_t batch) const {
    if (kind_ != Kind::Bluestein || sub_.three)
        return scratch_bytes(batch);
    uint32_t m = Mmin_.load(std::memory_order_relaxed); // (looked for on the first use)
    if (!m)
        Mmin_.store(m = var_.pow2_m ? blue_length(n_, prec_, false) : M_,
                    std::memory_order_relaxed);
    return (size_t)batch * m * elem_bytes(prec_) + 256;
}

uint64_t Plan1D::group_within(uint64_t batch, size_t room) const {
    uint64_t groups = 1;
    while (groups < batch && scratch_bytes((batch + groups - 1) / groups) > room)
        ++groups;
    return (batch + groups - 1) / groups;
}

size_t Plan1D::pass_inst_bytes() const {
    const uint32_t s = sub_.four    ? std::max(sub_.col.inst_stride, sub_.row.inst_stride)
                       : sub_.three ? sub_.col.inst_stride
                                    : sub_.direct.inst_stride;
    return (size_t)s * elem_bytes(prec_);
}

bool Plan1D::fuses_real_pre() const {
    if (kind_ != Kind::Direct || sub_.three || sub_.maxr != 16 ||
        (prec_ == 4 && split_dft_default()))
        return false;
    return sub_.four ? sub_.rq_row.p != nullptr : mixgen_len(sub_.L, prec_);
}

bool Plan1D::shaped_rows() const {
    return kind_ == Kind::Direct && !sub_.four && !sub_.three && fast_len(sub_.L) &&
           sub_.maxr >= 16;
}

// Bluestein with a three-pass inner length, one transform at a time as separate
// steps (the three-pass form has no fused convolution round):
//   y = pre(x): conj?(x[j]) chirp[j] for j < n, zeros up to M
//   y = DFT_M(y);  y = conj(y * FFT(h));  y = DFT_M(y)
//   X[k] = conj?(conj(y[k]) chirp[k] scale / M) for k < n
hipError_t Plan1D::bluestein_steps(const Layout& in, const Layout& out, uint64_t batch,
                                   bool inverse, double scale, void* scratch, hipStream_t s,
                                   uint32_t dft) const {
    const uint32_t M = sub_.L;
    if (in.C > 1 || out.C > 1 || in.inst || out.inst || out.real_post ||
        (in.flags & ~KFA_IO_REAL) || (out.flags & ~KFA_IO_REAL))
        return hipErrorInvalidValue;
    const size_t eb = elem_bytes(prec_);
    char* y = (char*)scratch;
    char* rest = y + ((size_t)M * eb + 255) / 256 * 256;
    const KfaIo yio = io_plain(y, M);
    const int ein = (in.flags & KFA_IO_REAL) ? 1 : 2, eout = (out.flags & KFA_IO_REAL) ? 1 : 2;
    for (uint64_t t = 0; t < batch; ++t) {
        const char* xp = (const char*)in.ptr + (int64_t)t * in.dist_hi * (int64_t)(eb / 2) * ein;
        char* op = (char*)out.ptr + (int64_t)t * out.dist_hi * (int64_t)(eb / 2) * eout;
        hipError_t e = launch_bluestein_pre(prec_, xp, in.stride, ein == 1, inverse, chirp_.p, y, n_,
                                            M, s);
        if (e == hipSuccess)
            e = sub_.run(yio, yio, 1.0, 1.0, 1, rest, s, false, dft);
        if (e == hipSuccess)
            e = launch_mul_conj(prec_, y, hhat_.p, M, s);
        if (e == hipSuccess)
            e = sub_.run(yio, yio, 1.0, 1.0, 1, rest, s, false, dft);
        if (e == hipSuccess)
            e = launch_bluestein_post(prec_, y, chirp_.p, op, out.stride, eout == 1, inverse,
                                      scale / (double)M, n_, s);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t Plan1D::execute(const Layout& in, const Layout& out, uint64_t batch, bool inverse,
                           double scale, void* scratch, hipStream_t s, const Fuse* fuse) const {
    if (batch == 0)
        return hipSuccess;
    const size_t eb = elem_bytes(prec_);
    KfaIo load = io_from(in), store = io_from(out);
    const bool scaled = scale != 1.0;
    if (out.real_post && (!(fuses_real_post() || fuses_real_post_shaped()) || inverse || scaled))
        return hipErrorInvalidValue;
    const uint32_t dft = (fuse && fuse->dft) ? fuse->dft : split_dft_default();
    if (kind_ == Kind::Identity || kind_ == Kind::Direct) {
        if (fuse && fuse->pw_in) {
            load.pw = (uint64_t)fuse->pw_in;
            load.flags |= KFA_IO_PW | KFA_IO_PW_LAYOUT | (fuse->pw_in_f64 ? KFA_IO_PW_F64 : 0);
            if (inverse)
                load.flags |= KFA_IO_CONJ2;
        } else if (inverse) {
            load.flags |= KFA_IO_CONJ1;
        }
        if (inverse)
            store.flags |= KFA_IO_CONJ2;
        if (scaled)
            store.flags |= KFA_IO_SCALE;
        return sub_.run(load, store, scale, 1.0, batch, scratch, s, fuse && fuse->onchip, dft);
    }
    if (fuse && fuse->pw_in)
        return hipErrorInvalidValue; // callers apply the product separately for these kinds
    const uint32_t L = sub_.L;
    char* sp = (char*)scratch;
    if (kind_ == Kind::Rader) {
        const bool real_in = (in.flags & KFA_IO_REAL) != 0;
        const bool real_out = (out.flags & KFA_IO_REAL) != 0;
        // one group of nb transforms on stream st, with x0, A[0] and the
        // convolution's scratch from gsp
        auto rader = [&](const Layout& gi, const Layout& go, uint64_t nb, char* gsp,
                         hipStream_t st) -> hipError_t {
            const KfaIo gl = io_from(gi), gs = io_from(go);
            void* x0 = gsp;
            gsp += ((nb * eb + 255) / 256) * 256;
            void* dc = gsp;
            gsp += ((nb * eb + 255) / 256) * 256;
            void* tmp = gsp;
            // out of place, the passes read x[0] where it lies; otherwise (the store
            // may reach another instance's) from a copy made before them
            const char *i0 = (const char*)gi.ptr, *o0 = (const char*)go.ptr;
            const uint64_t iu = eb / (real_in ? 2 : 1), ou = eb / (real_out ? 2 : 1);
            const bool rows = gl.C == 1 && gs.C == 1 && !gi.inst && !go.inst &&
                              gi.dist_hi >= 0 && go.dist_hi >= 0 && gl.stride == 1 &&
                              gs.stride == 1;
            const uint64_t ispan = ((nb - 1) * (uint64_t)gi.dist_hi + n_) * iu;
            const uint64_t ospan = ((nb - 1) * (uint64_t)go.dist_hi + n_) * ou;
            const bool apart = !recorder() && rows && (i0 + ispan <= o0 || o0 + ospan <= i0);
            hipError_t e = hipSuccess;
            if (!apart)
                e = launch_gather_first(prec_, real_in, gi.ptr, gi.dist_hi, gi.dist_lo,
                                        gi.C ? gi.C : 1, x0, nb, st, gi.inst);
            if (e != hipSuccess)
                return e;
            // one convolution: a[n] = x'[g^n], A = FFT_{p-1}(a) (A[0] saved to dc),
            // c = IFFT(A * FFT(b)); X[g^-m] = x0 + c[m]
            KfaIo l1 = gl;
            l1.flags |= KFA_IO_MAP | (inverse ? KFA_IO_CONJ1 : 0);
            l1.map = (uint64_t)qidx_.p;
            // both permutations stay inside positions [1, p) of an instance and the
            // scatter fills them
            l1.row_lo = 1;
            l1.row_span = n_;
            KfaIo s2 = gs;
            s2.flags |= KFA_IO_MAP | KFA_IO_CONJ1 | KFA_IO_SCALE | KFA_IO_ADDX0 |
                        (inverse ? KFA_IO_CONJ2 : 0) | (scaled ? KFA_IO_SCALE_POST : 0) |
                        (real_in ? KFA_IO_AUX_REAL : 0);
            s2.map = (uint64_t)pidx_.p;
            s2.row_lo = 1;
            s2.row_span = n_;
            s2.aux = apart ? (uint64_t)gi.ptr : (uint64_t)x0;
            s2.aux_dist = apart ? gi.dist_hi : (s2.C > 1) ? s2.C : 1; // (x0: instance hi*C + lo)
            s2.aux_dist_lo = (!apart && s2.C > 1) ? 1 : 0;
            // X[0] in the last pass's store where that pass is compiled for it
            // (a two-pass inner length: known before its first passes run)
            if (apart &&
                (!sub_.four ||
                 (rader_cols_len(sub_.N1) && sub_.maxr == 16 && !(prec_ == 4 && dft)))) {
                e = sub_.run_conv(l1, s2, 1.0 / (double)L, scale, nb, bhat_.p, hperm_.p, tmp, st,
                                  dc, dft, true);
                if (e != hipErrorNotSupported)
                    return e;
                (void)hipGetLastError();
            }
            e = sub_.run_conv(l1, s2, 1.0 / (double)L, scale, nb, bhat_.p, hperm_.p, tmp, st, dc,
                              dft);
            if (e != hipSuccess)
                return e;
            // X[0] = x0 + A[0] (x0 where it lies has the input's distance)
            if (apart)
                e = launch_gather_first(prec_, real_in, gi.ptr, gi.dist_hi, gi.dist_lo, 1, x0, nb,
                                        st, nullptr);
            if (e != hipSuccess)
                return e;
            return launch_rader_dc(prec_, x0, real_in, dc, 1, go.ptr, go.dist_hi, go.dist_lo,
                                   go.C ? go.C : 1, real_out, inverse, scale, nb, st, go.inst);
        };
        // a batch of long convolutions (two-pass inner length, 128 MiB or more) runs
        // as four groups alternating between the caller's stream and the side
        // stream, so that one group's passes run beside the other's; each stream
        // has its own part of the scratch (a one-pass convolution measured slower
        // in groups: 1009 x 16384, 0.33 against 0.31 ms)
        const uint64_t gb = (batch + 3) / 4;
        const size_t slot = 2 * (((size_t)gb * eb + 255) / 256) * 256 +
                            (((size_t)gb * L * eb + 255) / 256) * 256;
        const bool groups = tuning().pipe && !no_alloc() && !recorder() && sub_.four &&
                            batch >= 8 &&
                            (uint64_t)batch * L * eb >= ((uint64_t)128 << 20) && !in.inst &&
                            !out.inst && in.C <= 1 && out.C <= 1 &&
                            !(in.flags & ~KFA_IO_REAL) && !(out.flags & ~KFA_IO_REAL) &&
                            2 * slot <= scratch_bytes(batch);
        if (!groups)
            return rader(in, out, batch, sp, s);
        hipError_t e;
        hipStream_t side = fork_side(s, &e);
        if (e != hipSuccess)
            return e;
        const int64_t ib = (int64_t)(eb / 2) * ((in.flags & KFA_IO_REAL) ? 1 : 2);
        const int64_t ob = (int64_t)(eb / 2) * ((out.flags & KFA_IO_REAL) ? 1 : 2);
        uint64_t g = 0;
        for (uint64_t g0 = 0; g0 < batch; g0 += gb, ++g) {
            const bool odd = side && (g & 1);
            Layout gi = in, go = out;
            gi.ptr = (char*)in.ptr + (int64_t)g0 * in.dist_hi * ib;
            go.ptr = (char*)out.ptr + (int64_t)g0 * out.dist_hi * ob;
            e = rader(gi, go, std::min<uint64_t>(gb, batch - g0), sp + (odd ? slot : 0),
                      odd ? side : s);
            if (e != hipSuccess)
                return e;
        }
        return join_side(s, side);
    }
    // Bluestein: X = chirp . IDFT_M(DFT_M(chirp . x, zero padded) * FFT(h)) / M
    if (sub_.three)
        return bluestein_steps(in, out, batch, inverse, scale, scratch, s, dft);
    void* tmp = sp;
    KfaIo l1 = load;
    l1.flags |= KFA_IO_PW | (inverse ? KFA_IO_CONJ1 : 0);
    l1.pw = (uint64_t)chirp_.p;
    l1.valid = n_;
    KfaIo s2 = store;
    s2.flags |= KFA_IO_CONJ1 | KFA_IO_PW | KFA_IO_SCALE | (inverse ? KFA_IO_CONJ2 : 0);
    s2.pw = (uint64_t)chirp_.p;
    s2.valid = n_;
    return sub_.run_conv(l1, s2, scale / (double)L, 1.0, batch, hhat_.p, hperm_.p, tmp, s,
                         nullptr, dft);
}

// =============================================================== plan registry
// recursive: a three-pass plan's build asks the registry for its inner plan
static std::recursive_mutex g_reg_mu;
static std::map<std::tuple<uint32_t, int, uint32_t>, std::weak_ptr<Plan1D>> g_reg;

std::shared_ptr<Plan1D> get_plan(uint32_t n, int prec, PlanVariant v) {
    std::lock_guard<std::recursive_mutex> lk(g_reg_mu);
    auto key = std::make_tuple(n, prec, v.key());
    auto it = g_reg.find(key);
    if (it != g_reg.end()) {
        if (auto sp = it->second.lock())
            return sp;
    }
    auto p = std::make_shared<Plan1D>(n, prec, v);
    if (!p->build())
        return nullptr;
    g_reg[key] = p;
    return p;
}

bool ColumnConv::plan(uint32_t y_, int prec_) {
    prec = prec_;
    if (!colconv_len(y_) || !pass.plan(y_, prec))
        return false;
    y = y_;
    return true;
}

hipError_t ColumnConv::run(const void* a, void* b, bool blocked, uint64_t pitch, uint64_t cols,
                           double scale, hipStream_t s) const {
    ColConvArgs c;
    memset(&c, 0, sizeof(c));
    c.a = a;
    c.b = b;
    c.tw = pass.tw.p;
    c.pitch = pitch;
    c.cols = cols;
    c.blk = blocked ? 4ull * y : 0ull;
    c.scale = scale;
    c.xcds = xcd_tile_order();
    return prec == 8 ? launch_colconv_f64(y, c, s) : launch_colconv_f32(y, c, s);
}

bool make_real_twiddles(DevBuf& out, uint32_t h, int prec, bool inverse) {
    // st[i] = exp(-+ i pi ((i+1)/h + 1/2)) = exp(-+ 2 pi i (2(i+1) + h) / (4h))
    DevBuf t64;
    if (!t64.alloc((size_t)h * 16) || !out.alloc((size_t)h * elem_bytes(prec)))
        return false;
    std::vector<uint32_t> idx(h);
    for (uint32_t i = 0; i < h; ++i)
        idx[i] = (uint32_t)(((uint64_t)2 * (i + 1) + h) % (4ull * h));
    DevBuf d_idx;
    if (!d_idx.alloc((size_t)h * 4))
        return false;
    hipStream_t s = default_stream();
    if (!hip_ok(hipMemcpy(d_idx.p, idx.data(), (size_t)h * 4, hipMemcpyHostToDevice), "st idx"))
        return false;
    if (!hip_ok(launch_twiddle_indexed(t64.p, (const uint32_t*)d_idx.p, h, 4ull * h, inverse ? 1 : 0,
                                       s),
                "st"))
        return false;
    if (!hip_ok(launch_convert_from_f64(prec, out.p, t64.p, h, 1.0, s), "st convert"))
        return false;
    return hip_ok(hipStreamSynchronize(s), "st sync");
}

} // namespace kfa
