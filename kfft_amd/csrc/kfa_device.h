// Device-side building blocks of the transform engine: complex arithmetic,
// radix codelets and the fused element load/store operations of a pass.
#pragma once
#include <hip/hip_runtime.h>

#include "kfa_common.h"

namespace kfa {

// A device address that the arguments carry as an integer, as a pointer known to
// be global memory.  (A plain cast gives a generic pointer, whose accesses are
// FLAT instructions: they count on the LDS counter as well, so every LDS access
// after one waits for the memory round trip.)
template <typename P>
__device__ __forceinline__ P* gmem(uint64_t a) {
    typedef __attribute__((address_space(1))) P* GP;
    return (P*)(GP)a;
}

template <typename T>
struct alignas(2 * sizeof(T)) cx {
    T re, im;
};

template <typename T>
__device__ __forceinline__ cx<T> operator+(cx<T> a, cx<T> b) {
    return {a.re + b.re, a.im + b.im};
}
template <typename T>
__device__ __forceinline__ cx<T> operator-(cx<T> a, cx<T> b) {
    return {a.re - b.re, a.im - b.im};
}
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ cx<T> mul_mi(cx<T> a) { // a * (-i)
    return {a.im, -a.re};
}
template <typename T>
__device__ __forceinline__ cx<T> conj(cx<T> a) {
    return {a.re, -a.im};
}

// ---------------------------------------------------------------------------
// compile-time cos/sin of 2*pi*m/R: octant reduction on exact integers, then a
// Taylor series on |phi| <= pi/4
// ---------------------------------------------------------------------------
constexpr double kPi = 3.14159265358979323846264338327950288;

constexpr double taylor_sin(double x) {
    double t = x, s = x;
    for (int n = 1; n < 14; ++n) {
        t *= -x * x / ((2.0 * n) * (2.0 * n + 1));
        s += t;
    }
    return s;
}
constexpr double taylor_cos(double x) {
    double t = 1, s = 1;
    for (int n = 1; n < 14; ++n) {
        t *= -x * x / ((2.0 * n - 1) * (2.0 * n));
        s += t;
    }
    return s;
}
struct CS {
    double c, s;
};
constexpr CS cs_turn(long m, long R) {
    long u = (8 * (m % R) + 8 * R) % (8 * R); // angle = (pi/4) * u / R
    long o = u / R, rem = u % R;
    long quad = 0;
    double phi = 0;
    int sg = 1;
    if (o % 2 == 0) {
        quad = o / 2;
        phi = (kPi / 4) * (double)rem / (double)R;
        sg = 1;
    } else {
        quad = (o + 1) / 2;
        phi = (kPi / 4) * (double)(R - rem) / (double)R;
        sg = -1;
    }
    double cp = taylor_cos(phi), sp = taylor_sin(phi);
    double ca = 0, sa = 0;
    switch (quad % 4) {
    case 0: ca = 1; break;
    case 1: sa = 1; break;
    case 2: ca = -1; break;
    default: sa = -1; break;
    }
    return {ca * cp - sa * sg * sp, sa * cp + ca * sg * sp};
}
template <int R>
struct OddTab {
    double c[R], s[R];
    constexpr OddTab() : c(), s() {
        for (int m = 0; m < R; ++m) {
            CS v = cs_turn(m, R);
            c[m] = v.c;
            s[m] = v.s;
        }
    }
};

// ---------------------------------------------------------------------------
// radix codelets: forward DFT of v[0..R-1] in natural order, in place
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void dft4(cx<T>& a0, cx<T>& a1, cx<T>& a2, cx<T>& a3) {
    cx<T> s02 = a0 + a2, d02 = a0 - a2, s13 = a1 + a3, d13 = mul_mi(a1 - a3);
    a0 = s02 + s13;
    a2 = s02 - s13;
    a1 = d02 + d13;
    a3 = d02 - d13;
}

template <typename T, int R>
__device__ __forceinline__ void dft_odd(cx<T>* v) {
    constexpr int H = (R - 1) / 2;
    constexpr OddTab<R> tab{};
    cx<T> s[H + 1], d[H + 1];
    cx<T> y0 = v[0];
#pragma unroll
    for (int j = 1; j <= H; ++j) {
        s[j] = v[j] + v[R - j];
        d[j] = v[j] - v[R - j];
        y0 = y0 + s[j];
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        cx<T> ra = v[0], ia = {T(0), T(0)};
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const int m = (j * k) % R;
            const T c = (T)tab.c[m], sn = (T)tab.s[m];
            ra.re += s[j].re * c;
            ra.im += s[j].im * c;
            ia.re += d[j].re * sn;
            ia.im += d[j].im * sn;
        }
        v[k] = {ra.re + ia.im, ra.im - ia.re};
        v[R - k] = {ra.re - ia.im, ra.im + ia.re};
    }
    v[0] = y0;
}

template <typename T, int R>
__device__ __forceinline__ void dft(cx<T>* v) {
    if constexpr (R == 2) {
        cx<T> a = v[0], b = v[1];
        v[0] = a + b;
        v[1] = a - b;
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        const T r = (T)0.707106781186547524400844362104849039;
        cx<T> a0 = v[0], a1 = v[2], a2 = v[4], a3 = v[6];
        cx<T> b0 = v[1], b1 = v[3], b2 = v[5], b3 = v[7];
        dft4(a0, a1, a2, a3);
        dft4(b0, b1, b2, b3);
        b1 = {(b1.re + b1.im) * r, (b1.im - b1.re) * r};
        b2 = mul_mi(b2);
        b3 = {(b3.im - b3.re) * r, -(b3.re + b3.im) * r};
        v[0] = a0 + b0;
        v[4] = a0 - b0;
        v[1] = a1 + b1;
        v[5] = a1 - b1;
        v[2] = a2 + b2;
        v[6] = a2 - b2;
        v[3] = a3 + b3;
        v[7] = a3 - b3;
    } else if constexpr (R == 16) {
        const T c1 = (T)0.923879532511286756128183189396788933;
        const T s1 = (T)0.382683432365089771728459984030398866;
        const T r2 = (T)0.707106781186547524400844362104849039;
        cx<T> a[4][4]; // a[n2][k1]
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) {
            a[n2][0] = v[n2];
            a[n2][1] = v[4 + n2];
            a[n2][2] = v[8 + n2];
            a[n2][3] = v[12 + n2];
            dft4(a[n2][0], a[n2][1], a[n2][2], a[n2][3]);
        }
        // W16^(n2*k1)
        a[1][1] = cmul(a[1][1], cx<T>{c1, -s1});
        a[1][2] = cmul(a[1][2], cx<T>{r2, -r2});
        a[1][3] = cmul(a[1][3], cx<T>{s1, -c1});
        a[2][1] = cmul(a[2][1], cx<T>{r2, -r2});
        a[2][2] = mul_mi(a[2][2]);
        a[2][3] = cmul(a[2][3], cx<T>{-r2, -r2});
        a[3][1] = cmul(a[3][1], cx<T>{s1, -c1});
        a[3][2] = cmul(a[3][2], cx<T>{-r2, -r2});
        a[3][3] = cmul(a[3][3], cx<T>{-c1, s1});
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            cx<T> u0 = a[0][k1], u1 = a[1][k1], u2 = a[2][k1], u3 = a[3][k1];
            dft4(u0, u1, u2, u3);
            v[k1] = u0;
            v[k1 + 4] = u1;
            v[k1 + 8] = u2;
            v[k1 + 12] = u3;
        }
    } else {
        static_assert(R % 2 == 1, "unsupported even radix");
        dft_odd<T, R>(v);
    }
}

// ---------------------------------------------------------------------------
// fused load / store
// ---------------------------------------------------------------------------
struct Ctx {
    int64_t base;  // b_hi*dist_hi + b_lo*dist_lo
    uint32_t lo;   // b_lo
    uint32_t lgb;  // b_lo * lo_mul
    uint64_t hi;   // b_hi
};

template <uint32_t FM = KFA_IOM_ANY>
__device__ __forceinline__ Ctx make_ctx(const KfaIo& io, uint64_t inst) {
    Ctx c;
    uint64_t hi;
    uint32_t lo;
    if (io.C == 1) {
        hi = inst;
        lo = 0;
    } else if (inst <= 0xffffffffull) {
        const uint32_t i32 = (uint32_t)inst, h32 = i32 / io.C;
        hi = h32;
        lo = i32 - h32 * io.C;
    } else {
        hi = inst / io.C;
        lo = (uint32_t)(inst - hi * io.C);
    }
    c.base = ((io.flags & FM & KFA_IO_INST) ? gmem<const int64_t>(io.inst)[hi] : (int64_t)hi * io.dist_hi) +
             (int64_t)lo * io.dist_lo;
    c.lo = lo;
    c.lgb = lo * io.lo_mul;
    c.hi = hi;
    return c;
}

template <typename T>
__device__ __forceinline__ cx<T> pw_value(const KfaIo& io, uint32_t lg, int64_t addr) {
    const uint64_t idx = (io.flags & KFA_IO_PW_LAYOUT) ? (uint64_t)addr : (uint64_t)lg;
    if (io.flags & KFA_IO_PW_F64) {
        const cx<double> w = gmem<const cx<double>>(io.pw)[idx];
        return {(T)w.re, (T)w.im};
    }
    return gmem<const cx<T>>(io.pw)[idx];
}

template <typename T>
__device__ __forceinline__ cx<T> load_aux(const KfaIo& io, const Ctx& c) {
    const int64_t i = (int64_t)c.hi * io.aux_dist + (int64_t)c.lo * io.aux_dist_lo;
    if (io.flags & KFA_IO_AUX_REAL)
        return {gmem<const T>(io.aux)[i], T(0)};
    return gmem<const cx<T>>(io.aux)[i];
}

// ---------------------------------------------------------------------------
// A thread's elements of a pass move in batches: NB runs of R elements, run i at
// logical elements eb[i] + r * es (r < R), taking part where ok[i].  Every step
// (map, data, factor table, arithmetic, store) goes over the whole batch before
// the next one, with the step's flags tested once.  (Element by element, each
// load waits for the one before: the flag tests split the code into blocks, and
// a value's use in its block is a full memory round trip.)
// ---------------------------------------------------------------------------

// values held at a time by the steps that read one or two table entries per value
template <typename T>
constexpr int io_chunk() {
    return sizeof(T) == 8 ? 4 : 8;
}

// Element operations of a load on v[i R + r]: raw data from the instance in memory
// (LDS_ROW: from row[position], the instance's raw elements in LDS; lmap there
// holds a 16-bit copy of the map), 0 where the element is past the valid ones or
// does not take part.  Addresses advance by uniform steps from one per run: the
// 64-bit products per element cost more than the butterflies.
template <typename T, int NB, int R, bool LDS_ROW = false, uint32_t FM = KFA_IOM_ANY>
__device__ __forceinline__ void load_elems(const KfaIo& io, const Ctx& c, cx<T>* v,
                                           const uint32_t (&eb)[NB], const bool (&ok)[NB],
                                           uint32_t es, const cx<T>* row = nullptr,
                                           const uint16_t* lmap = nullptr) {
    const uint32_t fl = io.flags & FM;
    const bool map = (fl & KFA_IO_MAP) != 0, all = !(FM & KFA_IOM_PART) || io.valid == 0xffffffffu;
    const uint32_t ls = es * io.e_mul;              // logical step within a run
    const int64_t as = (int64_t)ls * io.stride;     // its address step (no map)
    uint32_t lg0[NB]; // first logical element of each run (runs that take no part: run 0 of
                      // lane 0, whose elements every instance has)
#pragma unroll
    for (int i = 0; i < NB; ++i)
        lg0[i] = c.lgb + (ok[i] ? eb[i] : 0u) * io.e_mul;
    auto lgi = [&](int i, int r) { return lg0[i] + (uint32_t)r * ls; };
    auto in = [&](int i, int r) { return ok[i] && (all || lgi(i, r) < io.valid); };
    const T one = (fl & KFA_IO_CONJ1) ? T(-1) : T(1);
    if constexpr (LDS_ROW) {
        // (positions of a generator map: read where the element takes part)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t lg = in(i, r) ? lgi(i, r) : 0u;
                const uint32_t ph = !map ? lg : lmap ? (uint32_t)lmap[lg]
                                                     : gmem<const uint32_t>(io.map)[lg];
                v[i * R + r] = row[ph];
            }
    } else {
        auto fetch = [&](auto raw) { // raw(address): the raw element there
            if (map) {
                const uint32_t* m = gmem<const uint32_t>(io.map);
                uint32_t ph[NB * R];
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        ph[i * R + r] = m[in(i, r) ? lgi(i, r) : 0u];
#pragma unroll
                for (int j = 0; j < NB * R; ++j)
                    v[j] = raw(c.base + (int64_t)ph[j] * io.stride);
            } else if (all) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int64_t a0 = c.base + (int64_t)lg0[i] * io.stride;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[i * R + r] = raw(a0 + r * as);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int64_t a0 = c.base + (int64_t)lg0[i] * io.stride;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        v[i * R + r] = {T(0), T(0)};
                        if (in(i, r))
                            v[i * R + r] = raw(a0 + r * as);
                    }
                }
            }
        };
        if (fl & KFA_IO_REAL)
            fetch([p = gmem<const T>(io.ptr)](int64_t a) { return cx<T>{p[a], T(0)}; });
        else
            fetch([p = gmem<const cx<T>>(io.ptr)](int64_t a) { return p[a]; });
    }
    if (fl & KFA_IO_PW) {
        constexpr int CH = io_chunk<T>();
        const bool lay = (fl & KFA_IO_PW_LAYOUT) != 0;
        // the factors' index: the logical element, or the data's address (no map)
        auto factors = [&](auto wat, int j0, cx<T>* w) {
#pragma unroll
            for (int k = 0; k < CH; ++k) {
                w[k] = {T(0), T(0)};
                if (j0 + k < NB * R) {
                    const int i = (j0 + k) / R, r = (j0 + k) % R;
                    if (in(i, r))
                        w[k] = wat(lay ? c.base + (int64_t)lg0[i] * io.stride + r * as
                                       : (int64_t)lgi(i, r));
                }
            }
        };
#pragma unroll
        for (int j0 = 0; j0 < NB * R; j0 += CH) {
            cx<T> w[CH];
            if (fl & KFA_IO_PW_F64)
                factors([p = gmem<const cx<double>>(io.pw)](int64_t x) {
                    const cx<double> d = p[x];
                    return cx<T>{(T)d.re, (T)d.im};
                }, j0, w);
            else
                factors([p = gmem<const cx<T>>(io.pw)](int64_t x) { return p[x]; }, j0, w);
            // (conjugation as a sign, so that no value is waited for before the first
            // factors are requested)
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (j0 + k < NB * R)
                    v[j0 + k] = cmul(cx<T>{v[j0 + k].re, v[j0 + k].im * one}, w[k]);
            __builtin_amdgcn_sched_barrier(0); // one chunk's factors held at a time
        }
    } else if (fl & KFA_IO_CONJ1) {
#pragma unroll
        for (int j = 0; j < NB * R; ++j)
            v[j].im = -v[j].im;
    }
    if (fl & KFA_IO_CONJ2) {
#pragma unroll
        for (int j = 0; j < NB * R; ++j)
            v[j].im = -v[j].im;
    }
    if (all) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (!ok[i])
                    v[i * R + r] = {T(0), T(0)};
    } else {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (!in(i, r))
                    v[i * R + r] = {T(0), T(0)};
    }
}

// write a stored value at position ph of the instance
template <typename T>
__device__ __forceinline__ void store_raw(const KfaIo& io, const Ctx& c, uint32_t ph, cx<T> v) {
    const int64_t addr = c.base + (int64_t)ph * io.stride;
    if (io.flags & KFA_IO_REAL) {
        gmem<T>(io.ptr)[addr] = v.re;
    } else if (io.flags & KFA_IO_REAL_PAIRS) {
        T* o = gmem<T>(io.ptr);
        o[c.base + (int64_t)(2 * ph) * io.stride] = v.re;
        o[c.base + (int64_t)(2 * ph + 1) * io.stride] = v.im;
    } else {
        gmem<cx<T>>(io.ptr)[addr] = v;
    }
}

// Element operations of a store on v[i R + r] (changed in place), then the store:
// to memory, or (LDS_ROW) to row[position] in LDS; lmap as for load_elems.
// Nothing is stored for elements past the valid ones.
template <typename T, int NB, int R, bool LDS_ROW = false, uint32_t FM = KFA_IOM_ANY>
__device__ __forceinline__ void store_elems(const KfaFftArgs& A, const Ctx& c, cx<T>* v,
                                            const uint32_t (&eb)[NB], const bool (&ok)[NB],
                                            uint32_t es, cx<T> x0, cx<T>* row = nullptr,
                                            const uint16_t* lmap = nullptr) {
    const KfaIo& io = A.out;
    constexpr int CH = io_chunk<T>();
    const uint32_t fl = io.flags & FM;
    const bool map = (fl & KFA_IO_MAP) != 0, all = !(FM & KFA_IOM_PART) || io.valid == 0xffffffffu;
    const uint32_t ls = es * io.e_mul;
    const int64_t as = (int64_t)ls * io.stride;
    uint32_t e0[NB], lg0[NB]; // (runs that take no part: element 0, unused)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        e0[i] = ok[i] ? eb[i] : 0u;
        lg0[i] = c.lgb + e0[i] * io.e_mul;
    }
    auto lgi = [&](int i, int r) { return lg0[i] + (uint32_t)r * ls; };
    auto in = [&](int i, int r) { return ok[i] && (all || lgi(i, r) < io.valid); };
    if (fl & KFA_IO_CONJ1) {
#pragma unroll
        for (int j = 0; j < NB * R; ++j)
            v[j].im = -v[j].im;
    }
    if (fl & KFA_IO_TW4) {
        // W_N^(b_lo * e) from two double tables; one rounding into T
        const cx<double>* th = gmem<const cx<double>>(A.tw4_hi);
        const cx<double>* tl = gmem<const cx<double>>(A.tw4_lo);
        const uint32_t lm = (1u << A.tw4_shift) - 1u;
        constexpr int TC = 4;
        const uint32_t ms = c.lo * es; // exponent step within a run
        uint32_t m0[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i)
            m0[i] = c.lo * e0[i];
#pragma unroll
        for (int j0 = 0; j0 < NB * R; j0 += TC) {
            cx<double> h[TC], l[TC];
#pragma unroll
            for (int k = 0; k < TC; ++k)
                if (j0 + k < NB * R) {
                    const int i = (j0 + k) / R, r = (j0 + k) % R;
                    const uint32_t m = m0[i] + (uint32_t)r * ms;
                    h[k] = th[m >> A.tw4_shift];
                    l[k] = tl[m & lm];
                }
#pragma unroll
            for (int k = 0; k < TC; ++k)
                if (j0 + k < NB * R) {
                    const cx<double> w = cmul(h[k], l[k]);
                    const cx<T> x = v[j0 + k];
                    v[j0 + k] = {(T)((double)x.re * w.re - (double)x.im * w.im),
                                 (T)((double)x.re * w.im + (double)x.im * w.re)};
                }
            __builtin_amdgcn_sched_barrier(0); // one chunk's table entries held at a time
        }
    }
    uint32_t ph[NB * R]; // positions (map only)
    if (map) {
        auto look = [&](auto m) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    ph[i * R + r] = m[in(i, r) ? lgi(i, r) : 0u];
        };
        if (LDS_ROW && lmap)
            look(lmap);
        else
            look(gmem<const uint32_t>(io.map));
    }
    if (fl & KFA_IO_PW) {
        const bool lay = (fl & KFA_IO_PW_LAYOUT) != 0;
#pragma unroll
        for (int j0 = 0; j0 < NB * R; j0 += CH) {
            cx<T> w[CH];
#pragma unroll
            for (int k = 0; k < CH; ++k) {
                w[k] = {T(0), T(0)};
                if (j0 + k < NB * R) {
                    const int i = (j0 + k) / R, r = (j0 + k) % R;
                    if (in(i, r))
                        w[k] = pw_value<T>(io, lgi(i, r),
                                           lay ? c.base + (int64_t)(map ? ph[j0 + k] : lgi(i, r)) *
                                                              io.stride
                                               : 0);
                }
            }
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (j0 + k < NB * R)
                    v[j0 + k] = cmul(v[j0 + k], w[k]);
            __builtin_amdgcn_sched_barrier(0); // one chunk's factors held at a time
        }
    }
    if (fl & KFA_IO_SCALE) {
        const T sc = (T)A.scale;
#pragma unroll
        for (int j = 0; j < NB * R; ++j) {
            v[j].re *= sc;
            v[j].im *= sc;
        }
    }
    if (fl & KFA_IO_CONJ2) {
#pragma unroll
        for (int j = 0; j < NB * R; ++j)
            v[j].im = -v[j].im;
    }
    if (fl & KFA_IO_ADDX0) {
#pragma unroll
        for (int j = 0; j < NB * R; ++j)
            v[j] = v[j] + x0;
    }
    if (fl & KFA_IO_SCALE_POST) {
        const T sc = (T)A.scale_post;
#pragma unroll
        for (int j = 0; j < NB * R; ++j) {
            v[j].re *= sc;
            v[j].im *= sc;
        }
    }
    if constexpr (LDS_ROW) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (in(i, r))
                    row[map ? ph[i * R + r] : lgi(i, r)] = v[i * R + r];
    } else {
        auto put = [&](auto raw) { // raw(address, value)
            if (map) {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (in(i, r))
                            raw(c.base + (int64_t)ph[i * R + r] * io.stride, v[i * R + r]);
            } else {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (!ok[i])
                        continue;
                    const int64_t a0 = c.base + (int64_t)lg0[i] * io.stride;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (all || lgi(i, r) < io.valid)
                            raw(a0 + r * as, v[i * R + r]);
                }
            }
        };
        if (fl & KFA_IO_REAL) {
            put([p = gmem<T>(io.ptr)](int64_t a, cx<T> x) { p[a] = x.re; });
        } else if (fl & KFA_IO_REAL_PAIRS) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (in(i, r))
                        store_raw<T>(io, c, map ? ph[i * R + r] : lgi(i, r), v[i * R + r]);
        } else {
            put([p = gmem<cx<T>>(io.ptr)](int64_t a, cx<T> x) { p[a] = x; });
        }
    }
}

template <typename T>
__device__ __forceinline__ uint32_t lds_index(uint32_t e) {
    return e + (e >> (sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32));
}

// Real-input rebuild of one bin pair (0 < k <= h/2) from Z = FFT_h(x as complex):
// f1 = Z[k] + conj(Z[h-k]), f2 = Z[k] - conj(Z[h-k]), t = f2 * st[k-1],
// X[k] = (f1 + t) / 2, X[h-k] = conj(f1 - t) / 2 (kfft_scalar.c:174-216).
template <typename T>
__device__ __forceinline__ void rebuild_pair(cx<T> za, cx<T> zb, cx<T> w, cx<T>& xk, cx<T>& xh) {
    const cx<T> bb = {zb.re, -zb.im};
    const cx<T> f1 = za + bb, f2 = za - bb;
    const cx<T> t = cmul(f2, w);
    xk = {(f1.re + t.re) * T(0.5), (f1.im + t.im) * T(0.5)};
    xh = {(f1.re - t.re) * T(0.5), (t.im - f1.im) * T(0.5)};
}

// Store of a pass carrying KFA_IO_RPOST: the instance's half-length spectrum Z
// (L values) is in LDS at z; bins X[0..L] of the real-input transform go to the
// output, lanes ln, ln + tpi, ... taking one pair (k, L-k) each.  X[0] and X[L]
// come from Z[0] with zero imaginary parts.
template <typename T>
__device__ __forceinline__ void store_real_post(const KfaIo& io, const Ctx& c, const cx<T>* z,
                                                uint32_t L, uint32_t ln, uint32_t tpi) {
    cx<T>* x = gmem<cx<T>>(io.ptr) + c.base;
    const int64_t xs = io.stride;
    const bool blk = (io.flags & KFA_IO_BLK4) != 0;
    auto at = [&](uint32_t k) {
        return blk ? (int64_t)(k >> 2) * xs + (k & 3u) : (int64_t)k * xs;
    };
    const cx<T>* st = gmem<const cx<T>>(io.pw);
    constexpr int CH = 4; // pairs at a time: their twiddle loads overlap
    for (uint32_t k0 = ln; k0 <= L / 2; k0 += CH * tpi) {
        cx<T> w[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t k = k0 + i * tpi;
            w[i] = st[(k >= 1 && k <= L / 2) ? k - 1 : 0u];
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t k = k0 + i * tpi;
            if (k == 0) {
                const cx<T> dc = z[lds_index<T>(0)];
                x[0] = {dc.re + dc.im, T(0)};
                x[at(L)] = {dc.re - dc.im, T(0)};
            } else if (k <= L / 2) {
                cx<T> xk, xh;
                rebuild_pair<T>(z[lds_index<T>(k)], z[lds_index<T>(L - k)], w[i], xk, xh);
                x[at(k)] = xk;
                x[at(L - k)] = xh;
            }
        }
    }
}

// Load of a pass carrying KFA_IO_RPRE: Z of the inverse rebuild
// (rebuild_inverse, kfft_scalar.c:218-242) from the instance's bins X[0..L] into
// LDS at z, lanes ln, ln + tpi, ... one pair (k, L - k) each:
//   Z[0] = (X[0] + X[L], X[0] - X[L]) of the real parts; with a = X[k] + conj
//   X[L-k], b = (X[k] - conj X[L-k]) st[k-1]:  Z[k] = a + b, Z[L-k] = conj(a - b)
template <typename T>
__device__ __forceinline__ void load_real_pre(const KfaIo& io, const Ctx& c, cx<T>* z, uint32_t L,
                                              uint32_t ln, uint32_t tpi) {
    const cx<T>* x = gmem<const cx<T>>(io.ptr) + c.base;
    const int64_t xs = io.stride;
    const bool blk = (io.flags & KFA_IO_BLK4) != 0;
    auto at = [&](uint32_t k) {
        return blk ? (int64_t)(k >> 2) * xs + (k & 3u) : (int64_t)k * xs;
    };
    const cx<T>* st = gmem<const cx<T>>(io.pw);
    constexpr int CH = 4; // pairs at a time: their loads overlap
    for (uint32_t k0 = ln; k0 <= L / 2; k0 += CH * tpi) {
        cx<T> xa[CH], xb[CH], w[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t k = k0 + i * tpi, kk = k <= L / 2 ? k : 0u;
            xa[i] = x[at(kk)];
            xb[i] = x[at(L - kk)];
            w[i] = st[kk ? kk - 1 : 0u];
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t k = k0 + i * tpi;
            if (k == 0) {
                z[lds_index<T>(0)] = {xa[i].re + xb[i].re, xa[i].re - xb[i].re};
            } else if (k <= L / 2) {
                const cx<T> fc = conj(xb[i]);
                const cx<T> a = xa[i] + fc, b = cmul(xa[i] - fc, w[i]), d = a - b;
                z[lds_index<T>(k)] = a + b;
                z[lds_index<T>(L - k)] = conj(d);
            }
        }
    }
}

} // namespace kfa
