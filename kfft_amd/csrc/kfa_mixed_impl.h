// Compile-time shaped FFT passes for mixed-radix lengths (2^a 3^b 5^c 7^d
// 11^e 13^f that fit one LDS pass), the counterpart of kfa_fast_impl.h's
// power-of-two passes.
//
// The radix sequence is the planner's (radix_list in kfa_engine.cpp with the
// default radix cap 16): radix-16 stages (or 16s then 8, 4), the 2 / 4 / 8
// remainder, 9s and a 3, then the odd primes in ascending order; so a pass
// shares the plan's stage-twiddle table (LdsPass layout).  Every thread owns up
// to 16 complex values: stage s runs NB(s) butterflies b = lane + i TPI per
// thread, masked where TPI NB(s) exceeds the stage's L / R(s) butterflies.
// Stage 0 loads straight from memory into registers, each stage boundary
// exchanges once through LDS, and the last stage stores from registers.
// Shapes, radices, thread counts and strides are template constants.
//
// Modes as in kfa_fast_impl.h: ROW (instances are rows), COL (lanes walk
// instances on both sides; optional W_N^(col e) on store), TOUT (load like
// ROW, store like COL).
#pragma once
#include "kfa_kernels.h"
#include "kfa_fast_impl.h"
#include "kfa_mix_sched.h"

namespace kfa {

// A tile-wide exchange of register values through LDS in two halves, the real
// parts and then the imaginary parts, so that an instance's LDS slot holds SP
// values of T instead of SP of cx<T>.  Register slot j takes part on the write
// (read) side where wok(j) (rok(j)), at position wpos(j) (rpos(j)) in T from m.
// A slot's imaginary part stays in its register until the second half, so the
// first half's reads may replace the real parts in place.
template <typename T, int E, class WO, class WP, class RO, class RP>
__device__ __forceinline__ void exchange_halves(cx<T>* v, T* m, WO wok, WP wpos, RO rok, RP rpos) {
    __syncthreads(); // every read of the exchange before is done
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (wok(j))
            m[wpos(j)] = v[j].re;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (rok(j))
            v[j].re = m[rpos(j)];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (wok(j))
            m[wpos(j)] = v[j].im;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j)
        if (rok(j))
            v[j].im = m[rpos(j)];
}

// Register slot j = i R + r of lane sl holds butterfly b = sl + i TPI of stage s
// (taking part while b < L / R(s)): its element at the stage's start is
// b + r L / R(s), at its end (b - k) R + k + r NS(s), k = b mod NS(s); the
// positions are padded as in every slot.
template <int L, int s>
__device__ __forceinline__ bool stage_ok(int j, uint32_t sl) {
    using M = Mix<L>;
    constexpr int R = M::R(s), NB = M::NB(s);
    return j / R < NB && (int)sl + (j / R) * M::TPI < L / R;
}
template <typename T, int L, int s>
__device__ __forceinline__ int stage_read_pos(int j, uint32_t sl) {
    using M = Mix<L>;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int R = M::R(s);
    const int e = (int)sl + (j / R) * M::TPI + (j % R) * (L / R);
    return e + (e >> PSH);
}
template <typename T, int L, int s>
__device__ __forceinline__ int stage_write_pos(int j, uint32_t sl) {
    using M = Mix<L>;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int R = M::R(s), NS = M::NS(s);
    const int b = (int)sl + (j / R) * M::TPI, k = b % NS;
    const int e = (b - k) * R + k + (j % R) * NS;
    return e + (e >> PSH);
}

// Stage s of a tile: LDS -> registers, twiddle (stages after the first), DFT_R(s),
// and (unless it is the last stage) registers -> LDS; then the stages after it.
// tw: the stage-twiddle table (LdsPass layout).  HX: the exchanges go through
// slots of T in two halves (exchange_halves), each one done at the end of the
// stage before, so a stage starts with its values already in registers; my is
// then the slot as T*.
template <typename T, int L, int s, bool PRE = false, bool HX = false>
__device__ __forceinline__ void mixed_stages(const cx<T>* twt, cx<T>* v, cx<T>* my, uint32_t sl) {
    using M = Mix<L>;
    static_assert(!(PRE && HX), "twiddle prefetch with the exchange in halves");
    if constexpr (s < M::S) {
        constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
        constexpr int R = M::R(s), NS = M::NS(s), NB = M::NB(s), STR = L / R, TPI = M::TPI;
        // PRE: the stage's twiddles are requested before the barrier (the values
        // of the stage before are in LDS, so their registers are free) and their
        // cache round trip overlaps the wait for the other waves
        const cx<T>* tw = twt + M::TWOFF(s);
        cx<T> wt[PRE && s > 0 ? M::E : 1];
        if constexpr (PRE && s > 0) {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)sl + i * TPI, k = b % NS;
                // (b past the stage's butterflies reads entry 0, unused)
#pragma unroll
                for (int r = 1; r < R; ++r)
                    wt[i * R + r] = tw[b < STR ? k * (R - 1) + r - 1 : 0];
            }
        }
        if constexpr (!HX) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)sl + i * TPI;
                if (b < STR) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int e = b + r * STR;
                        v[i * R + r] = my[e + (e >> PSH)];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int b = (int)sl + i * TPI, k = b % NS;
            if (s > 0 && b < STR) {
#pragma unroll
                for (int r = 1; r < R; ++r)
                    v[i * R + r] = cmul(v[i * R + r], PRE ? wt[PRE && s > 0 ? i * R + r : 0]
                                                          : tw[k * (R - 1) + r - 1]);
            }
            dft<T, R>(v + i * R);
        }
        if constexpr (s + 1 < M::S && HX) {
            exchange_halves<T, M::E>(
                v, reinterpret_cast<T*>(my), [&](int j) { return stage_ok<L, s>(j, sl); },
                [&](int j) { return stage_write_pos<T, L, s>(j, sl); },
                [&](int j) { return stage_ok<L, s + 1>(j, sl); },
                [&](int j) { return stage_read_pos<T, L, s + 1>(j, sl); });
        } else if constexpr (s + 1 < M::S) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)sl + i * TPI, k = b % NS;
                if (b < STR) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int e = (b - k) * R + k + r * NS;
                        my[e + (e >> PSH)] = v[i * R + r];
                    }
                }
            }
        }
        mixed_stages<T, L, s + 1, PRE, HX>(twt, v, my, sl);
    }
}

template <typename T, int L, int MODE, int IPW>
__device__ __forceinline__ void mixed_tile(const FastArgs& A, uint64_t first, cx<T>* lds) {
    using M = Mix<L>;
    static_assert(M::valid(), "length outside the mixed-radix passes");
    constexpr int E = M::E, TPI = M::TPI, NST = M::S;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (L + (L >> PSH)) | 1; // odd LDS stride per instance
    const uint32_t tid = threadIdx.x;
    const uint32_t li = (MODE == FAST_COL) ? tid % IPW : tid / TPI;
    const uint32_t ll = (MODE == FAST_COL) ? tid / IPW : tid % TPI;
    const uint32_t si = (MODE == FAST_ROW) ? tid / TPI : tid % IPW;
    const uint32_t sl = (MODE == FAST_ROW) ? tid % TPI : tid / IPW;

    cx<T> v[E];
    // ---- stage 0: memory -> registers, DFT_R0, registers -> LDS
    {
        constexpr int R = M::R(0), NB = M::NB(0), STR = L / R;
        const uint64_t inst = first + li;
        // threads past the batch read the tile's first instance and store nothing
        const uint64_t ld = inst < A.batch ? inst : first;
        const uint64_t hi = ld / A.in_C, lo = ld - hi * A.in_C;
        const cx<T>* p0 = (const cx<T>*)A.in + ((int64_t)hi * A.in_hi + (int64_t)lo * A.in_lo);
        const int64_t st = A.in_stride;
        // (one loop per cache policy: a per-load choice would issue both loads)
        auto load_all = [&](auto ld1) {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)ll + i * TPI;
                if (b < STR) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[i * R + r] = ld1(p0 + (int64_t)(b + r * STR) * st);
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[i * R + r] = {T(0), T(0)};
                }
            }
        };
        if (A.flags & KFA_FAST_NT_IN)
            load_all([](const cx<T>* p) { return load_nt(p); });
        else
            load_all([](const cx<T>* p) { return *p; });
        if (A.flags & KFA_FAST_CONJ_IN) {
#pragma unroll
            for (int k = 0; k < NB * R; ++k)
                v[k].im = -v[k].im;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
            dft<T, R>(v + i * R);
        if constexpr (NST > 1) {
            cx<T>* my = lds + (size_t)li * SP;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)ll + i * TPI;
                if (b < STR) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int e = b * R + r;
                        my[e + (e >> PSH)] = v[i * R + r];
                    }
                }
            }
        }
    }
    // ---- stages 1..NST-1 (their outputs stay in registers after the last)
    mixed_stages<T, L, 1, true>((const cx<T>*)A.tw, v, lds + (size_t)si * SP, sl);
    // ---- store: the last stage's outputs e = b + r (L / R_last), b < L / R_last
    {
        constexpr int RL = M::R(NST - 1), NB = M::NB(NST - 1), STR = L / RL;
        const uint32_t oi = (NST == 1) ? li : si, ol = (NST == 1) ? ll : sl;
        const uint64_t inst = first + oi;
        if (inst < A.batch) {
            const uint64_t hi = inst / A.out_C, lo = inst - hi * A.out_C;
            cx<T>* q0 = (cx<T>*)A.out + ((int64_t)hi * A.out_hi + (int64_t)lo * A.out_lo);
            const int64_t st = A.out_stride;
            const T sc = (T)A.scale;
            const bool scaled = (A.flags & KFA_FAST_SCALE) != 0;
            const bool cj = (A.flags & KFA_FAST_CONJ_OUT) != 0;
            const bool tw4 = (A.flags & (KFA_FAST_TW4 | KFA_FAST_TW4_HI)) != 0;
            // W_N^(col e) of a four-step pass A from the [k1][n2] table: col is the
            // instance's column (lo) in a 1D four-step, its row block (hi mod N2)
            // in a column four-step
            const bool by_hi = (A.flags & KFA_FAST_TW4_HI) != 0;
            const uint32_t ts = by_hi ? A.pad : A.out_C;
            const uint32_t col = by_hi ? (uint32_t)(hi % A.pad) : (uint32_t)lo;
            const cx<T>* w0 = (const cx<T>*)A.tw4 + col;
            auto store_all = [&](auto st1) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int b = (int)ol + i * TPI;
                    if (b < STR) {
#pragma unroll
                        for (int r = 0; r < RL; ++r) {
                            const int e = b + r * STR;
                            cx<T> x = v[i * RL + r];
                            if (tw4)
                                x = cmul(x, w0[(uint32_t)e * ts]);
                            if (scaled) {
                                x.re *= sc;
                                x.im *= sc;
                            }
                            if (cj)
                                x.im = -x.im;
                            st1(q0 + (int64_t)e * st, x);
                        }
                    }
                }
            };
            if (A.flags & KFA_FAST_NT_OUT)
                store_all([](cx<T>* p, cx<T> x) { store_nt(p, x); });
            else
                store_all([](cx<T>* p, cx<T> x) { *p = x; });
        }
    }
}

template <typename T, int L, int MODE, int IPW>
__global__ void __launch_bounds__(IPW* Mix<L>::TPI) k_mixed(const FastArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    uint32_t tile = blockIdx.x;
    if (A.xcds > 1) {
        const uint32_t n = A.xcds, G = gridDim.x, q = G / n, r = G - q * n;
        const uint32_t x = tile % n, j = tile / n;
        tile = x * q + (x < r ? x : r) + j;
    }
    mixed_tile<T, L, MODE, IPW>(A, (uint64_t)tile * IPW, reinterpret_cast<cx<T>*>(kfa_smem));
}

// instances per workgroup.  Rows: the count (within 512 threads and 64 KiB of
// LDS) whose workgroup wastes the smallest share of its last wave, at least 128
// threads where the LDS allows.  Columns: enough instances for 128-byte runs,
// within 1024 threads and 160 KiB.
template <typename T, int L, int MODE>
constexpr int mixed_ipw() {
    constexpr int TPI = Mix<L>::TPI;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int bytes = (int)sizeof(cx<T>) * ((L + (L >> PSH)) | 1);
    if (MODE == FAST_ROW) {
        int best = 1, best_u = -1;
        for (int ipw = 1; ipw * TPI <= 512 && (ipw == 1 || ipw * bytes <= 65536); ++ipw) {
            const int thr = ipw * TPI;
            int u = thr * 1000 / ((thr + 63) / 64 * 64); // lanes used, per mille
            if (thr < 128)
                u -= 200;
            if (u > best_u) {
                best = ipw;
                best_u = u;
            }
        }
        return best;
    }
    // columns: at least 128-byte runs (8 FP64 / 16 FP32 instances), then the
    // count within 512 threads and 80 KiB of LDS that uses the most lanes of
    // its waves (two such workgroups share a CU), the longest runs among equals
    constexpr int want = sizeof(T) == 8 ? 8 : 16;
    int best = 1, best_u = -1;
    for (int ipw = 1; ipw * TPI <= 512 && (ipw == 1 || ipw * bytes <= 80 * 1024); ++ipw) {
        const int thr = ipw * TPI;
        int u = thr * 1000 / ((thr + 63) / 64 * 64);
        if (ipw < want)
            u -= 500;
        if (u >= best_u) {
            best = ipw;
            best_u = u;
        }
    }
    return best;
}

template <typename T, int L, int MODE>
static hipError_t launch_mixed_t(const FastArgs& a, hipStream_t s) {
    constexpr int IPW = mixed_ipw<T, L, MODE>();
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (L + (L >> PSH)) | 1;
    constexpr uint32_t lds = Mix<L>::S > 1 ? (uint32_t)(IPW * SP * sizeof(cx<T>)) : 0u;
    static_assert(IPW * SP * sizeof(cx<T>) <= 160 * 1024, "LDS budget");
    static_assert(IPW * Mix<L>::TPI <= 1024, "workgroup size");
    // no real rebuild; no split-operand form (FP32; the FP64 passes ignore those
    // bits, as the power-of-two ones do)
    if ((a.flags & KFA_FAST_RPOST) ||
        (std::is_same<T, float>::value && (a.flags & (KFA_FAST_MFMA_F16 | KFA_FAST_MFMA_BF16))))
        return hipErrorNotSupported;
    static const hipError_t attr = [lds] {
        hipError_t e = hipFuncSetAttribute((const void*)k_mixed<T, L, MODE, IPW>,
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
    if (groups > 0x7fffffffull)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_mixed<T, L, MODE, IPW>), dim3((unsigned)groups),
                       dim3(IPW * Mix<L>::TPI), lds, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The same shaped stages behind the general pass's fused load and store
// operations (KfaFftArgs: gather / scatter maps, pointwise factors, four-step
// twiddles, scaling, x0 add, real input or output) and its convolution form:
// stage 0 reads its elements with load_elems straight from memory, the last
// stage writes them with store_elems straight from registers; a
// convolution pass (mid_pw) multiplies the first round's spectrum by its table
// and conjugates it in registers, then runs the stages again from LDS.  Threads
// walk the elements of an instance on the load (store) side, or, where that
// side's instances are adjacent in memory (in_jfast / out_jfast), the instances.
// A real-input rebuild in the store (KFA_IO_RPOST) stages the spectrum in LDS
// and rebuilds bin pairs (k, L - k) from there, as the general pass does.
// HX: every exchange in two halves through slots of SP values of T (half the
// LDS per instance); the launcher takes it only without row staging or rebuild.
// U: the use the tile is compiled for (KfaUse).  Bound by latency: a tile is a
// chain of dependent round trips (map or factors, data, stage twiddles, four-step
// factors), so its loads are batched (load_elems) and its registers set by use
// (mixgen_wpe).  Measured, whole transforms, element-by-element FLAT
// accesses in one tile for all uses -> this: 1009 x 16384 FP64 290 -> 275 us,
// 65537 x 256 FP64 724 -> 686, the forward real rows of a 4160^2 FP32 convolution
// 78 -> 52 (batched in a tile for all uses: 361, 643 and 62; 174 registers).  Then,
// with x[0] read and X[0] stored by the Rader passes themselves, rows staged eight
// elements at a time and the registers set by the LDS: 250 and 575, 257 x 60000 FP64
// 255 -> 141.  The gathered and scattered passes of 65537 are bound by their L2
// requests (16 bytes of each 128-byte line: the gather's texture-address units are busy
// 95% of the time, the scatter writes 2.5 times its output to memory).
template <typename T, int L, int IPW, bool HX = false, int U = KFA_USE_ANY>
__device__ __forceinline__ void mixgen_tile(const KfaFftArgs& A, uint64_t first, cx<T>* lds,
                                            uint32_t tid) {
    using M = Mix<L>;
    static_assert(M::valid(), "length outside the mixed-radix passes");
    constexpr uint32_t FI = kfa_use_in(U), FO = kfa_use_out(U);
    constexpr int CONV = U == KFA_USE_ANY ? -1 : kfa_use_conv(U) ? 1 : 0;
    constexpr int E = M::E, TPI = M::TPI, NST = M::S;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (L + (L >> PSH)) | 1;
    const uint32_t li = A.in_jfast ? tid % IPW : tid / TPI;
    const uint32_t ll = A.in_jfast ? tid / IPW : tid % TPI;
    const uint32_t si = A.out_jfast ? tid % IPW : tid / TPI;
    const uint32_t sl = A.out_jfast ? tid / IPW : tid % TPI;
    const uint32_t nin =
        (uint32_t)((A.batch - first) < (uint64_t)IPW ? (A.batch - first) : (uint64_t)IPW);
    const cx<T>* twt = gmem<const cx<T>>(A.tw);
    // KFA_IO_LMAP: 16-bit copies of the gather's and the scatter's maps behind the
    // instance slots (the launcher reserves them)
    uint16_t* const lmap = reinterpret_cast<uint16_t*>(lds + (size_t)IPW * SP);
    static_assert(!HX || NST > 1, "an exchange in halves needs two stages");
    T* const hx_lds = reinterpret_cast<T*>(lds); // HX: slot i at hx_lds + i * SP
    const bool lmaps = !HX && (A.in.flags & FI & KFA_IO_LMAP) && (A.in.flags & FI & KFA_IO_MAP) &&
                       (A.out.flags & FO & KFA_IO_MAP) && A.in.row_span &&
                       A.in.row_span <= (uint32_t)SP && A.in.stride == 1 && !A.in_jfast;

    cx<T> v[E];
    // ---- round 1, stage 0: the elements through load_elems, DFT_R0, -> LDS
    {
        constexpr int R = M::R(0), NB = M::NB(0), STR = L / R;
        const bool act = li < nin;
        const Ctx c = make_ctx<FI>(A.in, first + (act ? li : 0));
        uint32_t eb[NB];
        bool ok[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            eb[i] = ll + i * TPI;
            ok[i] = act && eb[i] < (uint32_t)STR;
        }
        // a gather (Rader's generator order) from rows that fit a slot: the rows
        // move to LDS contiguously, the permutation reads them there
        const bool stage_in = !HX && (A.in.flags & FI & KFA_IO_MAP) && A.in.row_span &&
                              A.in.row_span <= (uint32_t)SP && A.in.stride == 1 &&
                              !A.in_jfast;
        if constexpr (U == KFA_USE_RPRE) {
            cx<T>* row = lds + (size_t)li * SP;
            if (act)
                load_real_pre<T>(A.in, c, row, L, ll, TPI);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    cx<T> x = {T(0), T(0)};
                    if (ok[i])
                        x = row[lds_index<T>(eb[i] + (uint32_t)(r * STR))];
                    if (A.in.flags & KFA_IO_CONJ1)
                        x.im = -x.im;
                    v[i * R + r] = x;
                }
            __syncthreads(); // every read of the staged rows is done
        } else if (stage_in) {
            cx<T>* row = lds + (size_t)li * SP;
            // (eight elements, four map entries at a time: their loads overlap)
            constexpr int CH = 8, CM = 4;
            if (act)
                for (uint32_t q0 = A.in.row_lo + ll; q0 < A.in.row_span; q0 += CH * TPI) {
                    cx<T> x[CH];
                    auto each = [&](auto raw) {
#pragma unroll
                        for (int k = 0; k < CH; ++k) {
                            const uint32_t q = q0 + k * TPI;
                            x[k] = raw(c.base + (int64_t)(q < A.in.row_span ? q : A.in.row_lo));
                        }
                    };
                    if (A.in.flags & FI & KFA_IO_REAL)
                        each([p = gmem<const T>(A.in.ptr)](int64_t i) {
                            return cx<T>{p[i], T(0)};
                        });
                    else
                        each([p = gmem<const cx<T>>(A.in.ptr)](int64_t i) { return p[i]; });
#pragma unroll
                    for (int k = 0; k < CH; ++k) {
                        const uint32_t q = q0 + k * TPI;
                        if (q < A.in.row_span)
                            row[q] = x[k];
                    }
                }
            if (lmaps) // both maps beside the rows, for every instance
                for (uint32_t q0 = tid; q0 < (uint32_t)L; q0 += CM * IPW * TPI) {
                    uint32_t mi[CM], mo[CM];
#pragma unroll
                    for (int k = 0; k < CM; ++k) {
                        const uint32_t q = q0 + k * IPW * TPI;
                        mi[k] = gmem<const uint32_t>(A.in.map)[q < (uint32_t)L ? q : 0u];
                        mo[k] = gmem<const uint32_t>(A.out.map)[q < (uint32_t)L ? q : 0u];
                    }
#pragma unroll
                    for (int k = 0; k < CM; ++k) {
                        const uint32_t q = q0 + k * IPW * TPI;
                        if (q < (uint32_t)L) {
                            lmap[q] = (uint16_t)mi[k];
                            lmap[L + q] = (uint16_t)mo[k];
                        }
                    }
                }
            __syncthreads();
            load_elems<T, NB, R, true, FI>(A.in, c, v, eb, ok, STR, row, lmaps ? lmap : nullptr);
            __syncthreads(); // every read of the staged rows is done
        } else {
            load_elems<T, NB, R, false, FI>(A.in, c, v, eb, ok, STR);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
            dft<T, R>(v + i * R);
        if constexpr (HX) {
            // load-side lanes write, stage-side lanes read stage 1's values
            exchange_halves<T, E>(
                v, hx_lds, [&](int j) { return stage_ok<L, 0>(j, ll); },
                [&](int j) { return (int)li * SP + stage_write_pos<T, L, 0>(j, ll); },
                [&](int j) { return stage_ok<L, 1>(j, sl); },
                [&](int j) { return (int)si * SP + stage_read_pos<T, L, 1>(j, sl); });
        } else if constexpr (NST > 1) {
            cx<T>* my = lds + (size_t)li * SP;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int b = (int)ll + i * TPI;
                if (b < STR) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int e = b * R + r;
                        my[e + (e >> PSH)] = v[i * R + r];
                    }
                }
            }
        }
    }
    // (HX: the slot as T*, passed through the cx<T>* parameter, never read as cx<T>)
    cx<T>* my = HX ? reinterpret_cast<cx<T>*>(hx_lds + (size_t)si * SP) : lds + (size_t)si * SP;
    mixed_stages<T, L, 1, false, HX>(twt, v, my, sl);
    constexpr int RL = M::R(NST - 1), NBL = M::NB(NST - 1), STRL = L / RL;
    const uint32_t oi = (NST == 1) ? li : si, ol = (NST == 1) ? ll : sl;
    cx<T> a0 = {T(0), T(0)}; // ONE_RADER: A[0] of the instance, on its lane 0
    if constexpr (U == KFA_USE_ONE_RADER)
        a0 = v[0];
    // Rader's X[0] beside the scatter (lane 0 of an instance, its first tile)
    auto store_dc = [&](const Ctx& c, cx<T> x0, uint32_t lane) {
        if constexpr (U == KFA_USE_ONE_RADER || U == KFA_USE_A2_RADER) {
            if (A.dc_out && lane == 0 && c.lo == 0) {
                cx<T> d = U == KFA_USE_ONE_RADER ? a0 : gmem<const cx<T>>(A.dc_src)[c.hi];
                if (A.out.flags & KFA_IO_CONJ2)
                    d.im = -d.im;
                d = d + x0;
                if (A.out.flags & KFA_IO_SCALE_POST) {
                    d.re *= (T)A.scale_post;
                    d.im *= (T)A.scale_post;
                }
                if (A.out.flags & KFA_IO_REAL)
                    gmem<T>(A.out.ptr)[c.base] = d.re;
                else
                    gmem<cx<T>>(A.out.ptr)[c.base] = d;
            }
        }
    };
    // FP64: the product's factors held at a time (four: 1018 x 4000, 2048-point tiles,
    // 63.1 us against 62.3, 1999 x 2000, 4096 points, 71.1 and 69.8, shorter tiles alike)
    [[maybe_unused]] constexpr int MC = 8;
    // ---- convolution: spectrum times mid_pw, conjugated, then the stages again
    if (CONV != 0 && (CONV == 1 || A.mid_pw)) {
        const bool act = oi < nin;
        const uint64_t inst = first + oi;
        const uint64_t row = inst % A.mid_rows;
        const cx<T>* h = gmem<const cx<T>>(A.mid_pw) + row * L;
        if (A.mid_dc && act && row == 0 && ol == 0)
            gmem<cx<T>>(A.mid_dc)[inst / A.mid_rows] = v[0]; // element 0 (b = 0, r = 0)
        if constexpr (HX) {
            // the product in place, then natural order -> stage 0's values
#pragma unroll
            for (int i = 0; i < NBL; ++i) {
                const int b = (int)ol + i * TPI;
                if (b < STRL) {
#pragma unroll
                    for (int r = 0; r < RL; ++r) {
                        cx<T> x = cmul(v[i * RL + r], h[b + r * STRL]);
                        x.im = -x.im;
                        v[i * RL + r] = x;
                        if (sizeof(T) == 8 && (i * RL + r) % MC == MC - 1)
                            __builtin_amdgcn_sched_barrier(0); // MC factors held at a time
                    }
                }
            }
            // (the last stage's butterfly layout is its read layout: natural order)
            exchange_halves<T, E>(
                v, hx_lds + (size_t)si * SP, [&](int j) { return stage_ok<L, NST - 1>(j, ol); },
                [&](int j) { return stage_read_pos<T, L, NST - 1>(j, ol); },
                [&](int j) { return stage_ok<L, 0>(j, sl); },
                [&](int j) { return stage_read_pos<T, L, 0>(j, sl); });
        } else {
            cx<T>* mo = lds + (size_t)oi * SP;
            __syncthreads(); // the last stage's LDS reads are done
#pragma unroll
            for (int i = 0; i < NBL; ++i) {
                const int b = (int)ol + i * TPI;
                if (b < STRL) {
#pragma unroll
                    for (int r = 0; r < RL; ++r) {
                        const int e = b + r * STRL;
                        cx<T> x = cmul(v[i * RL + r], h[e]);
                        x.im = -x.im;
                        mo[e + (e >> PSH)] = x;
                        if (sizeof(T) == 8 && (i * RL + r) % MC == MC - 1)
                            __builtin_amdgcn_sched_barrier(0); // MC factors held at a time
                    }
                }
            }
        }
        mixed_stages<T, L, 0, false, HX>(twt, v, my, sl);
    }
    // ---- store: the elements through store_elems (after a second round the
    // values sit in the stage-side mapping, also for a one-stage length)
    const bool second = CONV < 0 ? A.mid_pw != 0 : CONV == 1;
    const uint32_t wi = second ? si : oi, wl = second ? sl : ol;
    if (!HX && (A.out.flags & FO & KFA_IO_RPOST)) {
        // the spectrum Z in natural order into LDS, then bins k and L - k of the
        // real-input spectrum from Z[k] and Z[L - k] (row mapping on this side)
        cx<T>* mo = lds + (size_t)wi * SP;
        __syncthreads(); // the last stage's LDS reads are done
#pragma unroll
        for (int i = 0; i < NBL; ++i) {
            const int b = (int)wl + i * TPI;
            if (b < STRL) {
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int e = b + r * STRL;
                    mo[e + (e >> PSH)] = v[i * RL + r];
                }
            }
        }
        __syncthreads();
        if (si < nin)
            store_real_post<T>(A.out, make_ctx(A.out, first + si), lds + (size_t)si * SP, L, sl,
                               TPI);
        return;
    }
    uint32_t eb[NBL];
    bool ok[NBL];
#pragma unroll
    for (int i = 0; i < NBL; ++i) {
        eb[i] = wl + i * TPI;
        ok[i] = eb[i] < (uint32_t)STRL;
    }
    // a scatter into rows that fit a slot: the values go to their positions in
    // LDS, then the rows leave contiguously ([row_lo, row_span) is filled)
    const bool stage_out = !HX && (A.out.flags & FO & KFA_IO_MAP) && A.out.row_span &&
                           A.out.row_span <= (uint32_t)SP && A.out.stride == 1 &&
                           !(A.out.flags & KFA_IO_REAL_PAIRS) && !A.out_jfast;
    if (stage_out) {
        cx<T>* row = lds + (size_t)wi * SP;
        __syncthreads(); // the last stage's LDS reads are done
        const Ctx c = make_ctx<FO>(A.out, first + (wi < nin ? wi : 0));
        if (wi < nin) {
            const cx<T> x0 =
                (A.out.flags & FO & KFA_IO_ADDX0) ? load_aux<T>(A.out, c) : cx<T>{T(0), T(0)};
            store_dc(c, x0, wl);
            store_elems<T, NBL, RL, true, FO>(A, c, v, eb, ok, STRL, x0, row,
                                              lmaps ? lmap + L : nullptr);
        }
        __syncthreads();
        if (wi < nin)
            for (uint32_t q = A.out.row_lo + wl; q < A.out.row_span; q += TPI)
                store_raw<T>(A.out, c, q, row[q]);
        return;
    }
    if (wi < nin) {
        const Ctx c = make_ctx<FO>(A.out, first + wi);
        const cx<T> x0 = (A.out.flags & FO & KFA_IO_ADDX0) ? load_aux<T>(A.out, c) : cx<T>{T(0), T(0)};
        store_dc(c, x0, wl);
        store_elems<T, NBL, RL, false, FO>(A, c, v, eb, ok, STRL, x0);
    }
}

// waves per SIMD a tile's registers are held to: FP64 tiles compiled for a use, what
// their LDS lets in, at most four (128 registers), three for the middle rows of a
// two-pass convolution, for Bluestein's passes and for Rader's scattered columns, which
// spill 10 to 90 registers at 128 (65537 x 256, middle rows, 102 us a group of 64
// transforms, 67 at 150 registers, the scattered columns 599 -> 584 the whole batch;
// 94132 x 44 280 -> 221 us, 2134 x 2000 346 -> 238, 1069 x 3923 170 -> 123, 254 x 16513
// 99 -> 65); the tile for all uses, what it needs (256 points at four waves spilled 136:
// 111 x 8000 real inverse 44 -> 30 us)
template <typename T, int L, int IPW, bool HX, int U>
constexpr int mixgen_wpe() {
    if (sizeof(T) == 4 || U == KFA_USE_ANY)
        return 1;
    constexpr int PSH = KFA_PAD_SHIFT_F64;
    constexpr int lds = IPW * ((L + (L >> PSH)) | 1) * (HX ? 8 : 16);
    constexpr int waves = (160 * 1024 / lds) * ((IPW * Mix<L>::TPI + 63) / 64) / 4;
    constexpr bool three = U == KFA_USE_MID || U == KFA_USE_ONE_BLUE || U == KFA_USE_A1_BLUE ||
                           U == KFA_USE_A2_BLUE || U == KFA_USE_A2_RADER;
    constexpr int most = three ? 3 : 4;
    return waves < 1 ? 1 : waves < most ? waves : most;
}
template <typename T, int L, int IPW, bool HX = false, int U = KFA_USE_ANY>
__global__ void __launch_bounds__(IPW* Mix<L>::TPI)
    __attribute__((amdgpu_waves_per_eu(mixgen_wpe<T, L, IPW, HX, U>()))) k_mixgen(const KfaFftArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    uint32_t tile = blockIdx.x;
    if (A.xcds > 1) {
        const uint32_t n = A.xcds, G = gridDim.x, q = G / n, r = G - q * n;
        const uint32_t x = tile % n, j = tile / n;
        tile = x * q + (x < r ? x : r) + j;
    }
    mixgen_tile<T, L, IPW, HX, U>(A, (uint64_t)tile * IPW, reinterpret_cast<cx<T>*>(kfa_smem),
                                  threadIdx.x);
}

// KFFT_AMD_MIX_HALVES (default 1): FP64 general-IO tiles without row staging or
// a rebuild exchange their values through LDS in two halves (0: whole values)
inline bool mix_halves() {
    static const bool on = [] {
        const char* e = getenv("KFFT_AMD_MIX_HALVES");
        return !e || atoi(e) != 0;
    }();
    return on;
}

constexpr bool prime_after(int L) { // L + 1 is prime
    for (int d = 2; d * d <= L + 1; ++d)
        if ((L + 1) % d == 0)
            return false;
    return true;
}
// the uses a length is compiled for (col: lanes walk instances): powers of two for
// Bluestein's passes (its default convolution lengths), rader_cols_len for the
// two-pass Rader convolution, every length for plain passes
template <int L, bool COL>
constexpr bool mixgen_use(int u) {
    constexpr bool p2 = (L & (L - 1)) == 0;
    switch (u) {
    case KFA_USE_PLAIN:
        return true;
    case KFA_USE_A1_BLUE:
    case KFA_USE_A2_BLUE:
        return p2 && L <= 1024 && COL;
    case KFA_USE_MID:
        return p2 && L <= 1024 && !COL;
    case KFA_USE_ONE_BLUE:
        return p2;
    case KFA_USE_RPRE:
        return !COL;
    case KFA_USE_A1_RADER:
    case KFA_USE_A2_RADER:
        return rader_cols_len(L) && COL;
    default:
        return false;
    }
}

// hipErrorNotSupported where the pass's radices are not Mix<L>'s (or a real
// rebuild would need the column mapping)
template <typename T, int L>
static hipError_t launch_mixgen_t(const KfaFftArgs& a, hipStream_t s) {
    using M = Mix<L>;
    // (the rebuild pairs bins across threads of one instance: row mapping)
    if (a.L != (uint32_t)L || a.nstages != (uint32_t)M::S ||
        ((a.out.flags & KFA_IO_RPOST) && a.out_jfast))
        return hipErrorNotSupported;
    for (int i = 0; i < M::S; ++i)
        if (a.st[i].radix != (uint32_t)M::R(i))
            return hipErrorNotSupported;
    const int use = kfa_use_of(a);
    auto go = [&](auto ipw_c, auto col_c) -> hipError_t {
        constexpr int IPW = decltype(ipw_c)::value;
        constexpr bool COL = decltype(col_c)::value;
        constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
        constexpr int SP = (L + (L >> PSH)) | 1;
        constexpr uint32_t lds = (uint32_t)(IPW * SP * sizeof(cx<T>));
        static_assert(IPW * SP * sizeof(cx<T>) <= 160 * 1024, "LDS budget");
        static_assert(IPW * M::TPI <= 1024, "workgroup size");
        // KFA_IO_LMAP: the two 16-bit maps (L entries each) behind the slots
        constexpr uint32_t lmb = (uint32_t)((4 * L + 15) / 16 * 16);
        constexpr bool lmap_fits = lds + lmb <= 160 * 1024;
        const uint64_t groups = (a.batch + IPW - 1) / IPW;
        if (!groups)
            return hipSuccess;
        if (groups > 0x7fffffffull)
            return hipErrorInvalidValue;
        // the kernel compiled for use u (hx: exchanges in halves) with `bytes` of LDS
        auto kernel = [&](auto u_c, auto hx_c, const KfaFftArgs& b, uint32_t bytes) -> hipError_t {
            constexpr int U = decltype(u_c)::value;
            constexpr bool HX = decltype(hx_c)::value;
            static const hipError_t attr = [] {
                hipError_t e =
                    hipFuncSetAttribute((const void*)k_mixgen<T, L, IPW, HX, U>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)(HX ? lds / 2 : lmap_fits ? lds + lmb : lds));
                if (e != hipSuccess)
                    (void)hipGetLastError(); // do not leave the error for the next launch
                return e;
            }();
            if (attr != hipSuccess)
                return attr;
            hipLaunchKernelGGL((k_mixgen<T, L, IPW, HX, U>), dim3((unsigned)groups),
                               dim3(IPW * M::TPI), bytes, s, b);
            return hipGetLastError();
        };
        // a gather and a scatter whose rows both move through LDS (Rader's
        // one-pass convolution) read their maps from LDS copies: the tile loads
        // them beside the rows, so no map read waits on the caches after that
        auto staged = [](const KfaIo& io, bool jfast) {
            return (io.flags & KFA_IO_MAP) && io.row_span && io.row_span <= (uint32_t)SP &&
                   io.row_span <= 65536u && io.stride == 1 && !jfast && io.C == 1 &&
                   io.e_mul == 1;
        };
        if (lmap_fits && staged(a.in, a.in_jfast) && staged(a.out, a.out_jfast) &&
            !(a.out.flags & (KFA_IO_REAL_PAIRS | KFA_IO_RPOST))) {
            KfaFftArgs b = a;
            b.in.flags |= KFA_IO_LMAP;
            if constexpr (!COL && prime_after(L)) {
                if (use == KFA_USE_ONE_RADER)
                    return kernel(std::integral_constant<int, KFA_USE_ONE_RADER>{},
                                  std::false_type{}, b, lds + lmb);
            }
            if (a.dc_out)
                return hipErrorNotSupported;
            return kernel(std::integral_constant<int, KFA_USE_ANY>{}, std::false_type{}, b,
                          lds + lmb);
        }
        // FP64 tiles whose rows do not move through LDS exchange in halves: half
        // the LDS per instance, so the VGPRs, not the LDS, set the workgroups per CU
        // (FP32 tiles, already at four or more waves per SIMD, measured slower in
        // halves: 65537 x 512 in the float build 1.06 against 1.02 ms)
        auto in_lds = [](const KfaIo& io, bool jfast) {
            return (io.flags & KFA_IO_MAP) && io.row_span && io.row_span <= (uint32_t)SP &&
                   io.stride == 1 && !jfast;
        };
        const bool halves = sizeof(T) == 8 && M::S > 1 && mix_halves() &&
                            !in_lds(a.in, a.in_jfast) &&
                            !(in_lds(a.out, a.out_jfast) && !(a.out.flags & KFA_IO_REAL_PAIRS)) &&
                            !(a.out.flags & KFA_IO_RPOST) && !(a.in.flags & KFA_IO_RPRE);
        auto form = [&](auto u_c) -> hipError_t {
            if constexpr (sizeof(T) == 8 && M::S > 1) {
                if (halves)
                    return kernel(u_c, std::true_type{}, a, lds / 2);
            }
            return kernel(u_c, std::false_type{}, a, lds);
        };
#define KFA_MIXGEN_USE(u)                                                                          \
    if constexpr (mixgen_use<L, COL>(u)) {                                                         \
        if (use == u)                                                                              \
            return form(std::integral_constant<int, u>{});                                         \
    }
        KFA_MIXGEN_USE(KFA_USE_PLAIN)
        KFA_MIXGEN_USE(KFA_USE_A1_BLUE)
        KFA_MIXGEN_USE(KFA_USE_MID)
        KFA_MIXGEN_USE(KFA_USE_A2_BLUE)
        KFA_MIXGEN_USE(KFA_USE_ONE_BLUE)
        KFA_MIXGEN_USE(KFA_USE_A1_RADER)
        KFA_MIXGEN_USE(KFA_USE_A2_RADER)
        KFA_MIXGEN_USE(KFA_USE_RPRE)
#undef KFA_MIXGEN_USE
        if ((a.in.flags & KFA_IO_RPRE) || a.dc_out)
            return hipErrorNotSupported; // (only their own tiles have that load, that store)
        return form(std::integral_constant<int, KFA_USE_ANY>{});
    };
    if (a.in_jfast || a.out_jfast)
        return go(std::integral_constant<int, mixed_ipw<T, L, FAST_COL>()>{}, std::true_type{});
    return go(std::integral_constant<int, mixed_ipw<T, L, FAST_ROW>()>{}, std::false_type{});
}

} // namespace kfa
