// Compile-time shaped FFT passes for power-of-two lengths 16..4096 (row passes
// also 8192).
//
// These carry the batched C2C hot path (one-pass transforms and both passes of
// a four-step transform).  Every thread owns E = 16 complex values (8 for
// L = 32): stage 0 loads them straight from HBM into registers, each stage
// boundary exchanges them once through LDS, and the last stage stores straight
// from registers to HBM.  Shapes, radices, thread counts and LDS strides are
// template constants, so the only runtime index arithmetic is the instance
// base address.
//
// Modes (thread -> work mapping on the load side / store side):
//   ROW   instance-major on both sides (contiguous rows, lanes walk elements)
//   COL   lanes walk instances on both sides (columns of a row-major matrix;
//         pass A of four-step, optional W_N^(col*k) twiddle on store)
//   TOUT  load like ROW, store like COL (pass B of four-step: the output
//         X[k1 + N1*k2] is contiguous across consecutive instances k1)
//   COLR  COL with the inverse of the real-input rebuild in the load (pass A of
//         an inverse real transform's half-length two-pass transform)
#pragma once
#include <stdlib.h>

#include <algorithm>

#include <type_traits>

#include "kfa_device.h"
#include "kfa_mfma.h"

namespace kfa {

enum { FAST_ROW = 0, FAST_COL = 1, FAST_TOUT = 2, FAST_COLR = 3 };

// radix sequence of radix_list() for L = 2^a: 16s, then 8 / 4 / 2 (or 8,4 for
// a = 4q+1, q > 0)
template <int L>
struct P2 {
    static constexpr int a = (L >= 8192) ? 13 : (L >= 4096) ? 12 : (L >= 2048) ? 11 : (L >= 1024) ? 10 : (L >= 512) ? 9
                           : (L >= 256) ? 8 : (L >= 128) ? 7 : (L >= 64) ? 6 : (L >= 32) ? 5 : 4;
    static constexpr int q = a / 4, rr = a % 4;
    static constexpr int S = (rr == 0) ? q : (rr == 1 && q > 0) ? q + 1 : q + 1;
    static constexpr int R(int s) {
        if (rr == 1 && q > 0) {
            if (s < q - 1)
                return 16;
            return s == q - 1 ? 8 : 4;
        }
        if (s < q)
            return 16;
        return rr == 1 ? 2 : rr == 2 ? 4 : 8;
    }
    static constexpr int NS(int s) { // product of the radices before stage s
        int p = 1;
        for (int i = 0; i < s; ++i)
            p *= R(i);
        return p;
    }
    static constexpr int TWOFF(int s) { // offset of stage s in the twiddle table
        int o = 0;
        for (int i = 1; i < s; ++i)
            o += NS(i) * (R(i) - 1);
        return o;
    }
    static constexpr int E = (L == 32) ? 8 : 16;
    static constexpr int TPI = L / E;
    static constexpr int PAD_L(int shift) { return L + (L >> shift); }
};

// streaming (non-temporal) element access, used to keep single-use input and
// output traffic from displacing data that is read again from the caches
template <typename T>
struct VecOf;
template <>
struct VecOf<float> {
    typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct VecOf<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};
template <typename T>
__device__ __forceinline__ cx<T> load_nt(const cx<T>* p) {
    typedef typename VecOf<T>::type V;
    const V v = __builtin_nontemporal_load(reinterpret_cast<const V*>(p));
    return {v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void store_nt(cx<T>* p, cx<T> x) {
    typedef typename VecOf<T>::type V;
    V v;
    v.x = x.re;
    v.y = x.im;
    __builtin_nontemporal_store(v, reinterpret_cast<V*>(p));
}

// One radix-R butterfly; radix-16 goes to the matrix cores when DK selects a
// split-operand form (FP32 data, whole waves only).
// (returns the split-FP16 codelet's range verdict, else false)
template <typename T, int R, int DK>
__device__ __forceinline__ bool dft_any(cx<T>* v, const MfmaConst<DK>& K, bool check = true) {
    if constexpr (R == 16 && DK != DFT_VALU && std::is_same<T, float>::value) {
        return dft16_mfma<DK>(v, K, check);
    } else {
        dft<T, R>(v);
        return false;
    }
}

// DFT kind a launch may use: the split forms need FP32 data and workgroups of
// whole waves (the matrix instruction spans all 64 lanes)
template <typename T, int L, int IPW, int DK>
constexpr int dft_kind() {
    return (DK != DFT_VALU && std::is_same<T, float>::value && (IPW * P2<L>::TPI) % 64 == 0)
               ? DK : DFT_VALU;
}

// Real-input rebuild in a transposing pass whose tile holds the rows of the
// half-length transform Z in LDS at their natural positions (row pairs a and
// N1 - a in slots j and j + IPW/2): X[k] from Z[k] and Z[h - k]
// (kfft_scalar.c:174-216), X[h] from Z[0]; h = N1 * L.  Thread (si, sl) writes
// the last stage's outputs e = sl + i TPI + r (L / R_last) of slot si (instance
// `inst`).
template <typename T, int L, int IPW>
__device__ __forceinline__ void rpost_rows(const FastArgs& A, const cx<T>* lds, uint32_t si,
                                           uint32_t sl, uint64_t inst) {
    using S = P2<L>;
    constexpr int NST = S::S, E = S::E, TPI = S::TPI;
    constexpr int RL = S::R(NST - 1), NB = E / RL, STR = L / RL;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (S::PAD_L(PSH)) | 1;
    const uint32_t n1 = A.out_C, half = IPW / 2;
    if (inst >= A.batch)
        return;
    const uint64_t hi = inst / n1;
    const uint32_t row = (uint32_t)(inst - hi * n1);
    const uint32_t ps = (row == 0 || row == n1 / 2) ? si : (si < half ? si + half : si - half);
    const cx<T>* my = lds + (size_t)si * SP;
    const cx<T>* mp = lds + (size_t)ps * SP;
    const cx<T> wa = ((const cx<T>*)A.rpost_st)[row]; // W_2h^row
    const cx<T>* we = (const cx<T>*)A.rpost_w2;        // W_2L^e
    cx<T>* q0 = (cx<T>*)A.out + ((int64_t)hi * A.out_hi + (int64_t)row * A.out_lo);
    // plain stores: the rows' halves run in opposite directions, and streaming
    // stores of such runs measured 9% slower
    auto put = [&](int64_t at, cx<T> x) { q0[at] = x; };
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const int e = (int)sl + i * TPI + r * STR;
            const cx<T> za = my[e + (e >> PSH)];
            if (row == 0 && e == 0) {
                put(0, {za.re + za.im, T(0)});
                put((int64_t)L * A.out_stride, {za.re - za.im, T(0)});
                continue;
            }
            const int pe = row == 0 ? L - e : L - 1 - e;
            const cx<T> zb = mp[pe + (pe >> PSH)];
            // st[k - 1] for k = row + N1 e: -i W_2h^row W_2L^e
            const cx<T> w = mul_mi(cmul(wa, we[e]));
            cx<T> xk, xh;
            rebuild_pair<T>(za, zb, w, xk, xh);
            put((int64_t)e * A.out_stride, xk);
        }
}

// (hi, lo) = divmod(first + j, C) for the instances j < IPW of one tile: the
// division of the tile's first instance once (uniform operands), then one
// compare per instance where IPW <= C < 2^31, a 32-bit division otherwise
// where C < 2^31 (hi and lo of a 64-bit instance index in general)
template <int IPW>
struct TileDiv {
    uint64_t q0;
    uint32_t r0, C;
    __device__ __forceinline__ TileDiv(uint64_t first, uint32_t c) {
        C = c;
        q0 = first / c;
        r0 = (uint32_t)(first - q0 * c);
    }
    __device__ __forceinline__ void at(uint32_t j, uint64_t& hi, uint64_t& lo) const {
        if (C >= (uint32_t)IPW && C < 0x80000000u) {
            const uint32_t l = r0 + j; // < 2C
            const bool w = l >= C;
            hi = q0 + (w ? 1u : 0u);
            lo = w ? l - C : l;
        } else if (C < 0x80000000u) {
            const uint32_t l = r0 + j, q = l / C;
            hi = q0 + q;
            lo = l - q * C;
        } else {
            const uint64_t i = q0 * C + r0 + j;
            hi = i / C;
            lo = i - hi * C;
        }
    }
};

// the column of the store twiddle table W_N^(col * e) for instance (hi, lo):
// lo in a 1D four-step, the row block hi mod N2 in a column four-step
__device__ __forceinline__ uint32_t tw4_col(const FastArgs& A, uint64_t hi, uint64_t lo) {
    if (A.flags & KFA_FAST_TW4_HI)
        return hi < 0x100000000ull ? (uint32_t)hi % A.pad : (uint32_t)(hi % A.pad);
    return (uint32_t)lo;
}

// W_N^m from the two short tables of KFA_FAST_TW4_SPLIT (m = col * k < N; column
// passes only)
template <typename T>
__device__ __forceinline__ cx<T> tw4_split(const FastArgs& A, uint32_t m) {
    const uint32_t sh = A.tw4_shift;
    return cmul(((const cx<T>*)A.tw4)[m >> sh], ((const cx<T>*)A.tw4_lo)[m & ((1u << sh) - 1u)]);
}

// Lengths whose every stage is radix 16 (16, 256, 4096).
template <int L>
constexpr bool all_radix16() {
    for (int s = 0; s < P2<L>::S; ++s)
        if (P2<L>::R(s) != 16)
            return false;
    return P2<L>::E == 16;
}

// One radix-16 stage of the split forms in the matrix layout: the lane holds the
// inputs x_{8h..8h+7} (h = lane / 32) of column c = lane mod 32 of both groups
// (xr / xi[g]) and receives the products' output rows (d[g]: Re y_{4h..4h+3},
// Re y_{8+4h..}, Im y_{4h..}, Im y_{8+4h..}), so no lane exchange surrounds the
// products.  The split-FP16 range handling is that of dft16_mfma, per
// butterfly: the two lanes holding a column combine their partial maxima with
// one lane swap, after which lane c has the maximum of column c of group 0 and
// lane 32 + c that of group 1.  Returns dft16_mfma's verdict.
template <int DK>
__device__ __forceinline__ bool mx_stage(float (&xr)[2][8], float (&xi)[2][8], kfa_f16v (&d)[2],
                                         const MfmaConst<DK>& K0, const MfmaConst<DK>& K1,
                                         bool check) {
    bool scaled = false, narrow = false;
    float sc[2] = {1.0f, 1.0f}, inv[2] = {1.0f, 1.0f};
    if constexpr (DK == DFT_SPLIT_F16) {
        if (check) {
            float m[2] = {0.0f, 0.0f};
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m[g]) : "v"(xr[g][i]), "v"(xi[g][i]));
            swap32(m[0], m[1]);
            const float full = fmaxf(m[0], m[1]);
            scaled = __any(!(full >= 0.5f && full < 16384.0f));
            narrow = !__any(!(full >= 0.5f && full <= 512.0f));
            if (scaled) {
                float f = 1.0f, fi = 1.0f; // this lane's column's factor and its inverse
                if (full > 0.0f) {
                    int e = ilogbf(full);
                    e = e > 120 ? 120 : (e < -110 ? -110 : e);
                    f = ldexpf(1.0f, 14 - e);
                    fi = ldexpf(1.0f, e - 14);
                }
                float a = f, b = f, ai = fi, bi = fi;
                swap32(a, b);
                swap32(ai, bi);
                sc[0] = a;
                sc[1] = b;
                inv[0] = ai;
                inv[1] = bi;
            }
        }
    }
    if (scaled) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                xr[g][i] *= sc[g];
                xi[g][i] *= sc[g];
            }
    }
    d[0] = mfma_dft_group<DK>(K0, xr[0], xi[0]);
    d[1] = mfma_dft_group<DK>(K1, xr[1], xi[1]);
    if (scaled) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int j = 0; j < 16; ++j)
                d[g][j] *= inv[g];
    }
    return narrow;
}

// output index of entry j < 8 of a lane's half of a column's outputs, and the
// entry's value (its real part is row j of the lane's result, its imaginary
// part row 8 + j)
__device__ __forceinline__ int mx_out_k(int j, uint32_t h) {
    return j < 4 ? 4 * (int)h + j : 8 + 4 * (int)h + (j - 4);
}
__device__ __forceinline__ cx<float> mx_out(const kfa_f16v& d, int j) {
    return cx<float>{d[j], d[8 + j]};
}

// Split-form tile (FP32 data) for lengths whose every stage is radix 16: the
// tile of fast_tile below with the same butterflies, LDS positions, twiddles and
// products (bit for bit the same results), but each lane keeps the matrix
// layout of mx_stage from the loads through LDS to the stores.  Lane c + 32 h
// of a wave works on the butterflies that threads wave + c and wave + 32 + c
// own in fast_tile (groups 0 and 1): it loads, reads and writes their elements
// 8h..8h+7 and stores their outputs y_{4h..4h+3}, y_{8+4h..8+4h+3}.
template <int L, int MODE, int IPW, int DK>
__device__ __forceinline__ void fast_tile_mx(const FastArgs& A, uint64_t first, cx<float>* lds) {
    typedef float T;
    using S = P2<L>;
    constexpr int TPI = S::TPI, NST = S::S, STR = L / 16;
    constexpr int PSH = KFA_PAD_SHIFT_F32;
    // LDS positions below split e + (e >> PSH) into a lane part and a constant
    // part: every constant term is a multiple of 16 (radix-16 strides)
    static_assert(PSH == 4, "LDS padding of one slot per 16 elements");
    constexpr int SP = (S::PAD_L(PSH)) | 1;
    auto pad = [](int e) { return e + (e >> 4); };
    const MfmaConst<DK> K = mfma_dft16_const<DK>();
    const uint32_t tid = threadIdx.x, h = (tid >> 5) & 1u;
    uint32_t li[2], ll[2], si[2], sl[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const uint32_t t = (tid & ~63u) + 32u * (uint32_t)g + (tid & 31u);
        li[g] = (MODE == FAST_COL) ? t % IPW : t / TPI;
        ll[g] = (MODE == FAST_COL) ? t / IPW : t % TPI;
        si[g] = (MODE == FAST_ROW) ? t / TPI : t % IPW;
        sl[g] = (MODE == FAST_ROW) ? t % TPI : t / IPW;
    }
    constexpr bool can_rpost = MODE == FAST_TOUT && NST > 1 && IPW >= 2 && IPW % 2 == 0;
    const bool rpost = can_rpost && (A.flags & KFA_FAST_RPOST) != 0;
    auto slot_inst = [&](uint32_t j) -> uint64_t { // as in fast_tile
        if (!rpost)
            return first + j;
        constexpr uint32_t half = IPW / 2 > 0 ? IPW / 2 : 1;
        const uint32_t n1 = A.out_C;
        const uint64_t b = first / n1;
        const uint32_t t = (uint32_t)(first - b * n1) / IPW;
        const uint32_t a = t * half + (j % half);
        const uint32_t row = j < half ? a : (a == 0 ? n1 / 2 : n1 - a);
        return b * n1 + row;
    };
    // output k of entry j: 4h + kk(j), kk(j) = j (j < 4) or 4 + j (j >= 4)
    auto kk = [](int j) { return j < 4 ? j : 4 + j; };
    // store twiddles held from the start: the FP16 256-point column pass of 32
    // or 64 instances (the other shapes, and BF16's three-term matrices, leave
    // no registers for them at their occupancy)
    constexpr bool pre_tw4 = MODE == FAST_COL && DK == DFT_SPLIT_F16 && L == 256 && IPW % 32 == 0;
    cx<T> w4[pre_tw4 ? 2 : 1][8];
    float xr[2][8], xi[2][8];
    kfa_f16v d[2];
    bool narrow0 = true, skip_check1 = false;
    // ---- stage 0: HBM -> registers, products, -> LDS (or HBM)
    {
        const int64_t st = A.in_stride;
        const cx<T>* p0[2];
        const TileDiv<IPW> din(first, A.in_C);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            uint64_t hi, lo;
            if (rpost) {
                const uint64_t inst = slot_inst(li[g]);
                const uint64_t ld = inst < A.batch ? inst : first;
                hi = ld / A.in_C;
                lo = ld - hi * A.in_C;
            } else {
                din.at(first + li[g] < A.batch ? li[g] : 0u, hi, lo);
            }
            p0[g] = (const cx<T>*)A.in +
                    ((int64_t)hi * A.in_hi + (int64_t)lo * A.in_lo +
                     ((int64_t)ll[g] + (int64_t)(8 * STR) * h) * A.in_stride);
        }
        if constexpr (pre_tw4) {
            if (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI)) {
                const bool by_hi = (A.flags & KFA_FAST_TW4_HI) != 0;
                const uint32_t ts = by_hi ? A.pad : A.out_C;
                const TileDiv<IPW> dout(first, A.out_C);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    uint64_t whi, wlo;
                    dout.at(first + si[g] < A.batch ? si[g] : 0u, whi, wlo);
                    const uint32_t col = tw4_col(A, whi, wlo);
                    const uint32_t k0 = (uint32_t)sl[g] + (uint32_t)(4 * STR) * h;
                    if (MODE == FAST_COL && (A.flags & KFA_FAST_TW4_SPLIT)) {
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            w4[pre_tw4 ? g : 0][j] =
                                tw4_split<T>(A, col * (k0 + (uint32_t)(kk(j) * STR)));
                    } else {
                        const cx<T>* w0 = (const cx<T>*)A.tw4 + (k0 * ts + col);
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            w4[pre_tw4 ? g : 0][j] = w0[(uint32_t)(kk(j) * STR) * ts];
                    }
                }
            }
        }
        cx<T> x[2][8];
        if (A.flags & KFA_FAST_NT_IN) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    x[g][i] = load_nt(p0[g] + (int64_t)(i * STR) * st);
        } else {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    x[g][i] = p0[g][(int64_t)(i * STR) * st];
        }
        if (A.flags & KFA_FAST_CONJ_IN) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    x[g][i].im = -x[g][i].im;
        }
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                xr[g][i] = x[g][i].re;
                xi[g][i] = x[g][i].im;
            }
        narrow0 = mx_stage<DK>(xr, xi, d, K, K, true);
        if constexpr (NST > 1) {
            // stage 0's butterfly b = ll writes element 16 b + k
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                cx<T>* my = lds + (size_t)li[g] * SP + pad((int)ll[g] * 16) + 4 * (int)h;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    my[kk(j)] = mx_out(d[g], j);
            }
        }
    }
    // ---- stages 1..NST-1: LDS -> registers, twiddle, products, -> LDS or HBM
#pragma unroll
    for (int s = 1; s < NST; ++s) {
        const int NS = S::NS(s);
        // the 256-point passes of 32 or 64 instances per tile: the stage's
        // twiddles W_256^(k r) are folded into the matrix (its variant k), since
        // the 32 butterflies of a group share k = sl mod 16 (transposing passes:
        // in the column passes the matrices beside the store twiddles measured
        // slower, and BF16's three-term ones cost a wave per SIMD)
        constexpr bool fold = L == 256 && MODE == FAST_TOUT && IPW % 32 == 0;
        MfmaConst<DK> Kt[fold ? 2 : 1];
        if constexpr (fold) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
                Kt[g] = mfma_const_at<DK, 16>(sl[g] % 16u);
        }
        const cx<T>* tw = (const cx<T>*)A.tw + S::TWOFF(s);
        cx<T> wt[2][8];
#pragma unroll
        for (int g = 0; g < 2 && !fold; ++g) {
            // r = 8h + i takes tw[k 15 + r - 1]; r = 0 (h = 0, i = 0) takes none
            // (and reads entry k 15, inside the table, unused)
            const cx<T>* tk = tw + ((int)sl[g] % NS) * 15 + 8 * (int)h;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                wt[g][i] = tk[i == 0 ? (h == 0 ? 0 : -1) : i - 1];
        }
        if (DK == DFT_SPLIT_F16 && s == 1)
            skip_check1 = !__syncthreads_or(narrow0 ? 0 : 1);
        else
            __syncthreads();
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            // element sl + r STR, r = 8h + i (STR a multiple of 16)
            const cx<T>* my = lds + (size_t)si[g] * SP + pad((int)sl[g]) +
                              8 * (int)h * (STR + STR / 16);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                cx<T> x = my[i * (STR + STR / 16)];
                if (!fold && !(i == 0 && h == 0))
                    x = cmul(x, wt[g][i]);
                xr[g][i] = x.re;
                xi[g][i] = x.im;
            }
        }
        if constexpr (fold)
            mx_stage<DK>(xr, xi, d, Kt[0], Kt[fold ? 1 : 0], !(s == 1 && skip_check1));
        else
            mx_stage<DK>(xr, xi, d, K, K, !(s == 1 && skip_check1));
        if (s + 1 < NST) {
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                // element (b - k) 16 + k + r NS, r = 4h + kk(j) (NS a multiple of 16)
                const int b = (int)sl[g], k = b % NS;
                cx<T>* my = lds + (size_t)si[g] * SP + pad((b - k) * 16 + k) +
                            4 * (int)h * (NS + NS / 16);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    my[kk(j) * (NS + NS / 16)] = mx_out(d[g], j);
            }
        }
    }
    // ---- real-input rebuild: the outputs to their natural positions in LDS
    if constexpr (can_rpost) {
        if (rpost) {
            __syncthreads(); // every read of the last stage's operands is done
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                cx<T>* my = lds + (size_t)si[g] * SP + pad((int)sl[g]) +
                            4 * (int)h * (STR + STR / 16);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    my[kk(j) * (STR + STR / 16)] = mx_out(d[g], j);
            }
            __syncthreads();
            const uint32_t osi = tid % IPW, osl = tid / IPW; // this thread's own slot
            rpost_rows<T, L, IPW>(A, lds, osi, osl, slot_inst(osi));
            return;
        }
    }
    // ---- store: outputs e = b + k (L / 16), b the butterfly of the last stage
    const TileDiv<IPW> dout(first, A.out_C);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const uint32_t oi = (NST == 1) ? li[g] : si[g], ol = (NST == 1) ? ll[g] : sl[g];
        if (first + oi >= A.batch)
            continue;
        uint64_t hi, lo;
        dout.at(oi, hi, lo);
        const int64_t st = A.out_stride;
        cx<T>* q0 = (cx<T>*)A.out + ((int64_t)hi * A.out_hi + (int64_t)lo * A.out_lo +
                                     ((int64_t)ol + (int64_t)(4 * STR) * h) * st);
        cx<T> y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            y[j] = mx_out(d[g], j);
        if (pre_tw4 && (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI))) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                y[j] = cmul(y[j], w4[pre_tw4 ? g : 0][j]);
        } else if (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI)) {
            const bool by_hi = (A.flags & KFA_FAST_TW4_HI) != 0;
            const uint32_t ts = by_hi ? A.pad : A.out_C;
            const uint32_t col = tw4_col(A, hi, lo);
            const uint32_t k0 = ol + (uint32_t)(4 * STR) * h;
            if (MODE == FAST_COL && (A.flags & KFA_FAST_TW4_SPLIT)) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    y[j] = cmul(y[j], tw4_split<T>(A, col * (k0 + (uint32_t)(kk(j) * STR))));
            } else {
                const cx<T>* w0 = (const cx<T>*)A.tw4 + (k0 * ts + col);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    y[j] = cmul(y[j], w0[(uint32_t)(kk(j) * STR) * ts]);
            }
        }
        if (A.flags & KFA_FAST_SCALE) {
            const T scl = (T)A.scale;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                y[j].re *= scl;
                y[j].im *= scl;
            }
        }
        if (A.flags & KFA_FAST_CONJ_OUT) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                y[j].im = -y[j].im;
        }
        if (A.flags & KFA_FAST_NT_OUT) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                store_nt(q0 + (int64_t)(kk(j) * STR) * st, y[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                q0[(int64_t)(kk(j) * STR) * st] = y[j];
        }
    }
}

// an entry of the inverse rebuild's table: a factor and what its rounding left
template <typename T>
struct RebuildRow {
    cx<T> hi;
    cx<float> lo;
};
static_assert(sizeof(RebuildRow<double>) == 32 && sizeof(RebuildRow<float>) == 16,
              "the planner's layout");

// Stage 0's inputs of column n2 of an inverse real transform's half-length
// transform: Z[k], k = n1 N2 + n2, from the bins X[0..h] of transform `hi`, h = L N2:
// with a = X[k] + conj X[h-k], d = X[k] - conj X[h-k], Z[k] = a + d i e^(i pi k / h)
// (rebuild_inverse, kfft_scalar.c:218-242), the factor from conj(W_2L^n1 W_2h^n2).
// rpost_st holds W_2L^n1, n1 < L, and what rounding took from it, rpost_w2 W_2h^n2 - 1,
// n2 < N2, which is small: the factor u + (lo + u d) is rounded once, as an entry of a
// whole table would be.  (The product of two rounded entries had 1.8 times its error,
// the transform 1.2% more, for 1% less time FP64 and up to 1% FP32, 4% at 2^21.)  Each
// bin is read by its own column's tile and by its partner's (N2 - n2), the second time
// from L2 (tiles of one transform share an XCD): inverse real 2^18 x 512 FP64 as part of
// a forward and inverse pass 2136 -> 1927 us against a rebuild sweep before the passes,
// 2^21 x 16 FP32 438 -> 383.
template <typename T, int L, int E>
__device__ __forceinline__ void rpre_column(const FastArgs& A, cx<T>* v, uint64_t hi, uint32_t n2,
                                            uint32_t ll) {
    using S = P2<L>;
    constexpr int R = S::R(0), STR = L / R, TPI = S::TPI;
    constexpr int CH = sizeof(T) == 8 ? 8 : 4; // bins at a time, with their partners
    const uint32_t N2 = A.in_C;
    const int64_t h = (int64_t)L * N2;
    const cx<T>* x = (const cx<T>*)A.in + (int64_t)hi * A.in_hi;
    const RebuildRow<T>* wr = (const RebuildRow<T>*)A.rpost_st;
    const cx<T> wd = ((const cx<T>*)A.rpost_w2)[n2];
#pragma unroll
    for (int j0 = 0; j0 < E; j0 += CH) {
        cx<T> xa[CH], xb[CH];
        RebuildRow<T> w[CH];
#pragma unroll
        for (int q = 0; q < CH; ++q) {
            const int i = (j0 + q) / R, r = (j0 + q) % R;
            const uint32_t n1 = ll + (uint32_t)(i * TPI + r * STR);
            const int64_t k = (int64_t)n1 * N2 + n2;
            xa[q] = x[k];
            xb[q] = x[h - k];
            w[q] = wr[n1];
        }
#pragma unroll
        for (int q = 0; q < CH; ++q) {
            const int i = (j0 + q) / R, r = (j0 + q) % R;
            const uint32_t n1 = ll + (uint32_t)(i * TPI + r * STR);
            if (n1 == 0 && n2 == 0)
                xa[q].im = xb[q].im = T(0); // (X[0] and X[h] count as real)
            const cx<T> f = conj(xb[q]), a = xa[q] + f, d = xa[q] - f;
            const cx<T> u = w[q].hi;
            const cx<T> W = {u.re + fma(-u.im, wd.im, fma(u.re, wd.re, (T)w[q].lo.re)),
                             u.im + fma(u.im, wd.re, fma(u.re, wd.im, (T)w[q].lo.im))};
            v[i * R + r] = a + cmul(d, cx<T>{W.im, W.re});
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One workgroup tile: instances [first, first + IPW) of the pass described by A.
// The caller provides the LDS area (IPW * SP elements).
template <typename T, int L, int MODE, int IPW, int DK = DFT_VALU>
__device__ __forceinline__ void fast_tile(const FastArgs& A, uint64_t first, cx<T>* lds) {
    using S = P2<L>;
    constexpr bool COLM = MODE == FAST_COL || MODE == FAST_COLR;
    constexpr int E = S::E, TPI = S::TPI, NST = S::S;
    constexpr int DKE = dft_kind<T, L, IPW, DK>();
    if constexpr (DKE != DFT_VALU && all_radix16<L>()) {
        fast_tile_mx<L, MODE, IPW, DKE>(A, first, lds);
        return;
    }
    MfmaConst<DKE> K;
    if constexpr (DKE != DFT_VALU)
        K = mfma_dft16_const<DKE>();
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (S::PAD_L(PSH)) | 1; // odd LDS stride per instance
    const uint32_t tid = threadIdx.x;
    // load side mapping
    const uint32_t li = (COLM) ? tid % IPW : tid / TPI;
    const uint32_t ll = (COLM) ? tid / IPW : tid % TPI;
    // store side (and middle stages) mapping
    const uint32_t si = (MODE == FAST_ROW) ? tid / TPI : tid % IPW;
    const uint32_t sl = (MODE == FAST_ROW) ? tid % TPI : tid / IPW;

    cx<T> v[E];
    // column passes of more than one stage hold their store twiddles from the
    // start where the registers allow it without costing occupancy: FP32 vector
    // stages, and the split-FP16 256-point column pass of 32 instances (measured:
    // the 2^16-point four-step 11% faster in FP32, 7% in split FP16; the FP64
    // passes and the other split shapes lose a wave per SIMD to it)
    constexpr bool pre_tw4 = MODE == FAST_COL && NST > 1 && sizeof(T) == 4 &&
                             (DKE == DFT_VALU || (DKE == DFT_SPLIT_F16 && L == 256 && IPW == 32));
    cx<T> w4[pre_tw4 ? E : 1];
    // split FP16: whether stage 0's inputs were narrow enough that stage 1 needs
    // no range test (decided for the whole workgroup at the first barrier)
    bool narrow0 = true, skip_check1 = false;
    // real-input rebuild (TOUT): slot j < IPW/2 of tile t of a transform holds
    // row a = t IPW/2 + j, slot j + IPW/2 its partner N1 - a (row N1/2 for a = 0),
    // so that every bin's partner bin h - k is in the workgroup (IPW divides N1)
    // (compiled only where a tile can hold row pairs; the launcher refuses the rest)
    constexpr bool can_rpost = MODE == FAST_TOUT && NST > 1 && IPW >= 2 && IPW % 2 == 0;
    const bool rpost = can_rpost && (A.flags & KFA_FAST_RPOST) != 0;
    auto slot_inst = [&](uint32_t j) -> uint64_t {
        if (!rpost)
            return first + j;
        constexpr uint32_t half = IPW / 2 > 0 ? IPW / 2 : 1;
        const uint32_t n1 = A.out_C;
        const uint64_t b = first / n1;
        const uint32_t t = (uint32_t)(first - b * n1) / IPW;
        const uint32_t a = t * half + (j % half);
        const uint32_t row = j < half ? a : (a == 0 ? n1 / 2 : n1 - a);
        return b * n1 + row;
    };
    // ---- stage 0: HBM -> registers, DFT_R0, registers -> LDS (or HBM)
    {
        constexpr int R = S::R(0), NB = E / R, STR = L / R;
        // threads past the batch read the tile's first instance (always valid) and
        // store nothing, so the loads need no per-element branches
        uint64_t hi, lo;
        if (rpost) {
            const uint64_t inst = slot_inst(li);
            const uint64_t ld = inst < A.batch ? inst : first;
            hi = ld / A.in_C;
            lo = ld - hi * A.in_C;
        } else {
            TileDiv<IPW>(first, A.in_C).at(first + li < A.batch ? li : 0u, hi, lo);
        }
        const cx<T>* p0 = (const cx<T>*)A.in +
                          ((int64_t)hi * A.in_hi + (int64_t)lo * A.in_lo + (int64_t)ll * A.in_stride);
        // the store's W_N^(col * e) factors (column passes): requested first, so
        // that their cache round trip overlaps the data's instead of following
        // the last stage, and waiting for the data implies them (every index stays
        // inside the [k1][n2] table: col < the table's row length for any
        // instance, e < L)
        if constexpr (pre_tw4) {
            if (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI)) {
                uint64_t whi, wlo;
                TileDiv<IPW>(first, A.out_C).at(first + si < A.batch ? si : 0u, whi, wlo);
                const bool by_hi = (A.flags & KFA_FAST_TW4_HI) != 0;
                const uint32_t ts = by_hi ? A.pad : A.out_C;
                const uint32_t col = tw4_col(A, whi, wlo);
                constexpr int RL = S::R(NST - 1), NBL = E / RL, STRL = L / RL;
                if (COLM && (A.flags & KFA_FAST_TW4_SPLIT)) {
#pragma unroll
                    for (int i = 0; i < NBL; ++i)
#pragma unroll
                        for (int r = 0; r < RL; ++r)
                            w4[i * RL + r] =
                                tw4_split<T>(A, col * ((uint32_t)sl + (uint32_t)(i * TPI + r * STRL)));
                } else {
                    const cx<T>* w0 = (const cx<T>*)A.tw4 + ((uint32_t)sl * ts + col);
#pragma unroll
                    for (int i = 0; i < NBL; ++i)
#pragma unroll
                        for (int r = 0; r < RL; ++r)
                            w4[i * RL + r] = w0[(uint32_t)(i * TPI + r * STRL) * ts];
                }
            }
        }
        const int64_t st = A.in_stride;
        if constexpr (MODE == FAST_COLR) {
            rpre_column<T, L, E>(A, v, hi, (uint32_t)lo, ll);
        } else if (A.flags & KFA_FAST_NT_IN) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[i * R + r] = load_nt(p0 + (int64_t)(i * TPI + r * STR) * st);
        } else {
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[i * R + r] = p0[(int64_t)(i * TPI + r * STR) * st];
        }
        if (A.flags & KFA_FAST_CONJ_IN) {
#pragma unroll
            for (int k = 0; k < E; ++k)
                v[k].im = -v[k].im;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
            narrow0 = dft_any<T, R, DKE>(v + i * R, K) && narrow0;
        if constexpr (NST > 1) {
            cx<T>* my = lds + (size_t)li * SP;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)ll + i * TPI;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int e = b * R + r;
                    my[e + (e >> PSH)] = v[i * R + r];
                }
            }
        }
    }
    // ---- stages 1..NST-1: LDS -> registers, twiddle, DFT, -> LDS or HBM
#pragma unroll
    for (int s = 1; s < NST; ++s) {
        const int R = S::R(s), NS = S::NS(s), NB = E / R, STR = L / R;
        // the stage's twiddles are requested before the barrier (the previous
        // stage's values are in LDS by now, so their registers are free), and
        // their cache round trip overlaps the wait for the other waves (not in
        // split-form passes that also hold their store twiddles: their matrix
        // operands leave no registers for both)
        constexpr bool pre_tw = DKE == DFT_VALU || !pre_tw4;
        const cx<T>* tw = (const cx<T>*)A.tw + S::TWOFF(s);
        cx<T> wt[E];
        auto load_tw = [&] {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)sl + i * TPI, k = b % NS;
#pragma unroll
                for (int r = 1; r < R; ++r)
                    wt[i * R + r] = tw[k * (R - 1) + r - 1];
            }
        };
        if (pre_tw)
            load_tw();
        if (DKE == DFT_SPLIT_F16 && s == 1 && S::R(0) == 16)
            skip_check1 = !__syncthreads_or(narrow0 ? 0 : 1);
        else
            __syncthreads();
        cx<T>* my = lds + (size_t)si * SP;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int e = (int)sl + i * TPI + r * STR;
                v[i * R + r] = my[e + (e >> PSH)];
            }
        if (!pre_tw)
            load_tw();
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 1; r < R; ++r)
                v[i * R + r] = cmul(v[i * R + r], wt[i * R + r]);
        // R is a compile-time constant after unrolling over s
        if (R == 16) {
#pragma unroll
            for (int i = 0; i < E / 16; ++i)
                dft_any<T, 16, DKE>(v + i * 16, K, !(s == 1 && skip_check1));
        } else if (R == 8) {
#pragma unroll
            for (int i = 0; i < E / 8; ++i)
                dft<T, 8>(v + i * 8);
        } else if (R == 4) {
#pragma unroll
            for (int i = 0; i < E / 4; ++i)
                dft<T, 4>(v + i * 4);
        } else {
#pragma unroll
            for (int i = 0; i < E / 2; ++i)
                dft<T, 2>(v + i * 2);
        }
        if (s + 1 < NST) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)sl + i * TPI, k = b % NS;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int e = (b - k) * R + k + r * NS;
                    my[e + (e >> PSH)] = v[i * R + r];
                }
            }
        }
    }
    // ---- real-input rebuild: the rows' Z through LDS, then X[k] from Z[k] and
    // Z[h - k]
    if constexpr (can_rpost) {
        if (rpost) {
            constexpr int RL = S::R(NST - 1), NB = E / RL, STR = L / RL;
            __syncthreads(); // every read of the last stage's operands is done
            cx<T>* my = lds + (size_t)si * SP;
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int e = (int)sl + i * TPI + r * STR;
                    my[e + (e >> PSH)] = v[i * RL + r];
                }
            __syncthreads();
            rpost_rows<T, L, IPW>(A, lds, si, sl, slot_inst(si));
            return;
        }
    }
    // ---- store: last stage outputs e = b + r * (L / R_last) (b < L / R_last)
    {
        constexpr int RL = S::R(NST - 1), NB = E / RL, STR = L / RL;
        const uint32_t oi = (NST == 1) ? li : si, ol = (NST == 1) ? ll : sl;
        if (first + oi < A.batch) {
            uint64_t hi, lo;
            TileDiv<IPW>(first, A.out_C).at(oi, hi, lo);
            cx<T>* q0 = (cx<T>*)A.out + ((int64_t)hi * A.out_hi + (int64_t)lo * A.out_lo +
                                         (int64_t)ol * A.out_stride);
            const int64_t st = A.out_stride;
            if (pre_tw4 && (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI))) {
#pragma unroll
                for (int k = 0; k < E; ++k)
                    v[k] = cmul(v[k], w4[pre_tw4 ? k : 0]);
            } else if (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI)) {
                // W_N^(col * e) from the [k1][n2] table: col is the instance's column
                // (lo) in a 1D four-step, its row block (hi mod N2) in a column four-step
                const bool by_hi = (A.flags & KFA_FAST_TW4_HI) != 0;
                const uint32_t ts = by_hi ? A.pad : A.out_C;
                const uint32_t col = tw4_col(A, hi, lo);
                if (COLM && (A.flags & KFA_FAST_TW4_SPLIT)) {
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int r = 0; r < RL; ++r)
                            v[i * RL + r] = cmul(v[i * RL + r],
                                                 tw4_split<T>(A, col * ((uint32_t)ol +
                                                                        (uint32_t)(i * TPI + r * STR))));
                } else {
                    const cx<T>* w0 = (const cx<T>*)A.tw4 + ((uint32_t)ol * ts + col);
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int r = 0; r < RL; ++r)
                            v[i * RL + r] =
                                cmul(v[i * RL + r], w0[(uint32_t)(i * TPI + r * STR) * ts]);
                }
            }
            if (A.flags & KFA_FAST_SCALE) {
                const T sc = (T)A.scale;
#pragma unroll
                for (int k = 0; k < E; ++k) {
                    v[k].re *= sc;
                    v[k].im *= sc;
                }
            }
            if (A.flags & KFA_FAST_CONJ_OUT) {
#pragma unroll
                for (int k = 0; k < E; ++k)
                    v[k].im = -v[k].im;
            }
            if (A.flags & KFA_FAST_NT_OUT) {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int r = 0; r < RL; ++r)
                        store_nt(q0 + (int64_t)(i * TPI + r * STR) * st, v[i * RL + r]);
            } else {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int r = 0; r < RL; ++r)
                        q0[(int64_t)(i * TPI + r * STR) * st] = v[i * RL + r];
            }
        }
    }
}

__device__ __forceinline__ uint32_t fast_tile_of(const FastArgs& A) {
    uint32_t tile = blockIdx.x;
    if (A.xcds > 1) {
        const uint32_t n = A.xcds, G = gridDim.x, q = G / n, r = G - q * n;
        const uint32_t x = tile % n, j = tile / n;
        tile = x * q + (x < r ? x : r) + j;
    }
    return tile;
}

// COLR tiles: registers held to what the LDS lets in (four FP32 waves per SIMD)
template <typename T, int L, int IPW>
__global__ void __launch_bounds__(IPW* P2<L>::TPI)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2))) k_fast_colr(const FastArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    // tiles of a transform from both ends in turn: a tile's partner bins are the
    // columns of the tile as far from the other end
    uint32_t tile = fast_tile_of(A);
    const uint32_t nt = A.in_C / IPW; // (both powers of two, IPW <= in_C)
    if (nt > 1) {
        const uint32_t j = tile & (nt - 1);
        tile = tile - j + ((j & 1) ? nt - 1 - (j >> 1) : j >> 1);
    }
    fast_tile<T, L, FAST_COLR, IPW>(A, (uint64_t)tile * IPW, reinterpret_cast<cx<T>*>(kfa_smem));
}

template <typename T, int L, int MODE, int IPW, int DK>
__global__ void __launch_bounds__(IPW* P2<L>::TPI) k_fast(const FastArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    const uint32_t tile = fast_tile_of(A);
    fast_tile<T, L, MODE, IPW, DK>(A, (uint64_t)tile * IPW, reinterpret_cast<cx<T>*>(kfa_smem));
}

template <int L, int MODE, typename T, int MUL>
constexpr int fast_ipw() {
    // instances per workgroup: ~256 threads for row passes; column passes take
    // enough instances for >= 128-byte runs (times MUL), capped by threads and LDS
    constexpr int TPI = P2<L>::TPI;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int bytes = (int)sizeof(cx<T>) * ((P2<L>::PAD_L(PSH)) | 1); // per instance
    constexpr int thr = (1024 / TPI) > 0 ? (1024 / TPI) : 1;
    // widened column tiles (MUL > 1) may fill the CU's LDS, except at 1024
    // points, where two workgroups of at most 80 KiB per CU (a power of two of
    // instances) are faster (measured: the 1024 x 1024 two-pass transform 23%
    // faster; 512-point transposing passes are faster with one full workgroup)
    constexpr int lim = MUL == 1 ? 65536 : (L >= 1024 ? 80 * 1024 : 160 * 1024);
    constexpr int fit = lim / bytes > 0 ? lim / bytes : 1;
    constexpr int cap = (MUL == 1 || L < 1024) ? fit : (fit >= 16 ? 16 : fit >= 8 ? 8
                                                        : fit >= 4 ? 4 : fit >= 2 ? 2 : 1);
    if (MODE == FAST_ROW) {
        constexpr int want = 256 / TPI > 0 ? 256 / TPI : 1;
        constexpr int c1 = (65536 / bytes) > 0 ? (65536 / bytes) : 1;
        return want < c1 ? want : c1;
    }
    constexpr int want = (sizeof(T) == 8 ? 8 : 16) * MUL;
    constexpr int w = want < cap ? want : cap;
    return w < thr ? w : thr;
}

template <typename T, int L, int MODE, int IPW, int DK>
constexpr auto fast_kernel() {
    if constexpr (MODE == FAST_COLR)
        return k_fast_colr<T, L, IPW>;
    else
        return k_fast<T, L, MODE, IPW, DK>;
}

template <typename T, int L, int MODE, int MUL, int DK>
static hipError_t launch_fast_t(const FastArgs& a, hipStream_t s) {
    constexpr int IPW = fast_ipw<L, MODE, T, MUL>();
    constexpr int DKE = dft_kind<T, L, IPW, DK>();
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (P2<L>::PAD_L(PSH)) | 1;
    const uint32_t lds = P2<L>::S > 1 ? (uint32_t)(IPW * SP * sizeof(cx<T>)) : 0u;
    static_assert(IPW * SP * sizeof(cx<T>) <= 160 * 1024, "LDS budget");
    static_assert(IPW * P2<L>::TPI <= 1024, "workgroup size");
    // the rebuild pairs rows a and N1 - a inside one tile
    // (whole transforms, no other store operations)
    if ((a.flags & KFA_FAST_RPOST) &&
        (MODE != FAST_TOUT || P2<L>::S < 2 || IPW < 2 || IPW % 2 || a.out_C % IPW ||
         a.batch % a.out_C ||
         (a.flags & (KFA_FAST_CONJ_OUT | KFA_FAST_SCALE | KFA_FAST_TW4 | KFA_FAST_TW4_HI))))
        return hipErrorNotSupported;
    // exactly the dynamic LDS it uses (a kernel with static LDS, a workgroup
    // reduction, cannot be granted the whole 160 KiB as dynamic LDS); set once
    // per process, thread-safe as a function-local static's initialisation
    static const hipError_t attr = [lds] {
        hipError_t e = hipFuncSetAttribute((const void*)fast_kernel<T, L, MODE, IPW, DKE>(),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)std::max<uint32_t>(lds, 1u));
        if (e != hipSuccess)
            (void)hipGetLastError(); // do not leave the error for the next launch
        return e;
    }();
    if (attr != hipSuccess)
        return attr;
    const uint64_t groups = (a.batch + IPW - 1) / IPW;
    if (!groups)
        return hipSuccess;
    hipLaunchKernelGGL((fast_kernel<T, L, MODE, IPW, DKE>()), dim3((unsigned)groups),
                       dim3(IPW * P2<L>::TPI), lds, s, a);
    return hipGetLastError();
}

// column-pass width multiplier (1, 2 or 4; default 2, measured), fixed per process
// (KFFT_AMD_COLS_MUL)
static inline int fast_cols_mul() {
    static const int m = [] {
        const char* e = getenv("KFFT_AMD_COLS_MUL");
        const int v = e ? atoi(e) : 2;
        return (v == 2 || v == 4) ? v : 1;
    }();
    return m;
}

template <typename T, int L, int MODE, int DK>
static hipError_t launch_fast_sel(const FastArgs& a, hipStream_t s) {
    if constexpr (MODE != FAST_ROW && L >= 64 && L <= 1024) {
        const int m = fast_cols_mul();
        if (m == 2)
            return launch_fast_t<T, L, MODE, 2, DK>(a, s);
        if (m == 4)
            return launch_fast_t<T, L, MODE, 4, DK>(a, s);
    }
    return launch_fast_t<T, L, MODE, 1, DK>(a, s);
}

// instances per workgroup of the transposing pass of length L (as launched)
template <typename T, int L>
static uint32_t tout_ipw_t() {
    if constexpr (L >= 64 && L <= 1024) {
        const int m = fast_cols_mul();
        if (m == 2)
            return (uint32_t)fast_ipw<L, FAST_TOUT, T, 2>();
        if (m == 4)
            return (uint32_t)fast_ipw<L, FAST_TOUT, T, 4>();
    }
    return (uint32_t)fast_ipw<L, FAST_TOUT, T, 1>();
}

template <typename T>
static uint32_t fast_tout_ipw_any(uint32_t L) {
    switch (L) {
    case 16: return tout_ipw_t<T, 16>();
    case 32: return tout_ipw_t<T, 32>();
    case 64: return tout_ipw_t<T, 64>();
    case 128: return tout_ipw_t<T, 128>();
    case 256: return tout_ipw_t<T, 256>();
    case 512: return tout_ipw_t<T, 512>();
    case 1024: return tout_ipw_t<T, 1024>();
    case 2048: return tout_ipw_t<T, 2048>();
    case 4096: return tout_ipw_t<T, 4096>();
    default: return 0;
    }
}

template <typename T, int MODE, int DK>
static hipError_t launch_fast_mode(uint32_t L, const FastArgs& a, hipStream_t s) {
    switch (L) {
    case 16: return launch_fast_sel<T, 16, MODE, DK>(a, s);
    case 32: return launch_fast_sel<T, 32, MODE, DFT_VALU>(a, s); // radices 8, 4
    case 64: return launch_fast_sel<T, 64, MODE, DK>(a, s);
    case 128: return launch_fast_sel<T, 128, MODE, DK>(a, s);
    case 256: return launch_fast_sel<T, 256, MODE, DK>(a, s);
    case 512: return launch_fast_sel<T, 512, MODE, DK>(a, s);
    case 1024: return launch_fast_sel<T, 1024, MODE, DK>(a, s);
    case 2048: return launch_fast_sel<T, 2048, MODE, DK>(a, s);
    case 4096: return launch_fast_sel<T, 4096, MODE, DK>(a, s);
    case 8192:
        if constexpr (MODE == FAST_ROW) // one instance per workgroup: rows only
            return launch_fast_sel<T, 8192, MODE, DK>(a, s);
        return hipErrorNotSupported;
    default: return hipErrorNotSupported;
    }
}

// column passes with the inverse rebuild in the load (vector stages)
template <typename T>
static hipError_t launch_fast_colr(uint32_t L, const FastArgs& a, hipStream_t s) {
    switch (L) {
    case 64: return launch_fast_t<T, 64, FAST_COLR, 2, DFT_VALU>(a, s);
    case 128: return launch_fast_t<T, 128, FAST_COLR, 2, DFT_VALU>(a, s);
    case 256: return launch_fast_t<T, 256, FAST_COLR, 2, DFT_VALU>(a, s);
    case 512: return launch_fast_t<T, 512, FAST_COLR, 2, DFT_VALU>(a, s);
    case 1024: return launch_fast_t<T, 1024, FAST_COLR, 2, DFT_VALU>(a, s);
    default: return hipErrorNotSupported;
    }
}

template <typename T, int DK>
static hipError_t launch_fast_dk(uint32_t L, int mode, const FastArgs& a, hipStream_t s) {
    if (mode == FAST_COL)
        return launch_fast_mode<T, FAST_COL, DK>(L, a, s);
    if (mode == FAST_TOUT)
        return launch_fast_mode<T, FAST_TOUT, DK>(L, a, s);
    return launch_fast_mode<T, FAST_ROW, DK>(L, a, s);
}

// KFA_FAST_MFMA_F16 / KFA_FAST_MFMA_BF16 in a.flags select the split-operand
// radix-16 stages (FP32 only; the FP64 passes always run on the vector units)
template <typename T>
static hipError_t launch_fast_any(uint32_t L, int mode, const FastArgs& a, hipStream_t s) {
    if (mode == FAST_COLR)
        return launch_fast_colr<T>(L, a, s);
    if constexpr (std::is_same<T, float>::value) {
        if (a.flags & KFA_FAST_MFMA_F16)
            return launch_fast_dk<T, DFT_SPLIT_F16>(L, mode, a, s);
        if (a.flags & KFA_FAST_MFMA_BF16)
            return launch_fast_dk<T, DFT_SPLIT_BF16>(L, mode, a, s);
    }
    return launch_fast_dk<T, DFT_VALU>(L, mode, a, s);
}

} // namespace kfa
