// The batched LDS-resident FFT pass, templated on precision and on the most
// complex values a thread holds per stage (MAXE).
//
// A workgroup owns `ipw` consecutive instances of a length-L transform.
//  1. Load: tpi threads per instance, each walking elements lane, lane + tpi,
//     ...; the lanes of one instance sit on consecutive threads (row passes) or
//     the same lane of consecutive instances does (in_jfast, column passes).
//     The pass's fused load operations apply on the way into a padded LDS
//     region per instance; plain layouts advance one address per element.
//  2. Radix stages, LDS to LDS, `tpi` threads per instance (Stockham autosort):
//       stage s of radix R, ns = product of earlier radices, butterfly b < L/R:
//         x_r = lds[b + r L/R] * W_{ns R}^{r (b mod ns)}
//         y   = DFT_R(x)
//         lds[(b - b mod ns) R + (b mod ns) + r ns] = y_r
//     A thread reads all of its butterflies, the workgroup synchronises, then
//     it computes and writes them back.
//  3. Store with the fused store operations, threads mapped like the load
//     (by out_jfast); or, for KFA_IO_RPOST, the real-input rebuild of bin
//     pairs (k, L-k) read from LDS.
// The DFT computed is always the forward one (negative exponent); inverse
// transforms conjugate on the way in and out.  A convolution pass (Bluestein,
// mid_pw) multiplies the spectrum by a table and conjugates it between two
// rounds of the stages, so its store sees conj(DFT(conj(DFT(x) * h))).
#pragma once
#include <type_traits>

#include "kfa_device.h"
#include "kfa_mfma.h"
#include "kfa_mix_sched.h"

namespace kfa {

// IO of a stage: LDS to LDS, or (the last stage of a plain row layout) LDS to
// memory.  "Plain": element e at base + (lgb + e e_mul) stride, complex or real,
// with at most conjugation and scaling (fused_io_plain).  (Reading stage 0's
// inputs from memory the same way spilled registers of the pass.)
enum { ST_LDS = 0, ST_OUT = 2 };

__device__ __forceinline__ bool fused_io_plain(const KfaIo& io, uint32_t extra) {
    return (io.flags & ~(KFA_IO_REAL | KFA_IO_CONJ1 | KFA_IO_CONJ2 | KFA_IO_INST | extra)) == 0 &&
           io.valid == 0xffffffffu;
}

// DK (FP32 only): radix-16 stages as split FP16 / BF16 matrix products
// (kfa_mfma.h).  The matrix instruction spans the wave, so in such a stage
// every lane runs the DFT of each of its butterfly slots, idle slots on zeros,
// while the loads, twiddles and stores stay masked.
// LC != 0: the pass's length is the compile-time LC and this is its stage SI
// (Mix<LC> schedule): butterfly counts, strides and twiddle offsets are
// constants; LC == 0: they come from the arguments.
template <typename T, int R, int MAXE, int IO = ST_LDS, int DK = DFT_VALU, int LC = 0, int SI = 0,
          bool PRE = true>
__device__ __forceinline__ void lds_stage(const KfaFftArgs& A, uint32_t s, cx<T>* my, uint32_t lane,
                                          bool act, const cx<T>* ltw, const MfmaConst<DK>& K,
                                          uint64_t inst = 0) {
    constexpr bool CT = LC != 0;
    using M = Mix<(CT ? LC : 1)>;
    constexpr int NB = CT ? M::NB(SI) : ((MAXE / R) > 0 ? (MAXE / R) : 1);
    constexpr bool MF = DK != DFT_VALU && R == 16 && std::is_same<T, float>::value;
    const uint32_t nb = CT ? (uint32_t)(LC / R) : A.L / R;
    const uint32_t ns = CT ? (uint32_t)M::NS(SI) : A.st[s].ns;
    const uint32_t tpi = CT ? (uint32_t)M::TPI : A.tpi;
    const uint32_t tw_off = CT ? (uint32_t)M::TWOFF(SI) : A.st[s].tw_off;
    const uint32_t magic = CT ? 0u : A.st[s].ns_magic;
    // b mod ns with b, ns < 2^16 (the LDS pass lengths): one multiply-high (a
    // constant divisor where the length is compiled in)
    auto mod_ns = [&](uint32_t b) { return CT ? b % ns : b - __umulhi(b, magic) * ns; };
    cx<T> v[NB][R];
    // the stage twiddles do not depend on LDS: in FP32 (radix <= 16) their
    // loads are issued first so that their latency overlaps the LDS reads and
    // the barrier (FP64 and the large prime radices would spill the registers
    // they hold across the barrier)
    constexpr bool early = PRE && sizeof(T) == 4 && R <= 16;
    // FP64 up to radix 16: twiddles through a generic pointer, whose loads the compiler
    // keeps apart.  As global loads they are all requested before the products, and with
    // eight elements loaded at a time the pass then spilled 34 registers (2 in this form).
    // 4 million points FP64, global loads and eight elements -> generic and six: 1287
    // points 92.0 -> 70.5 us, 858 69.7 -> 55.2, 135 54.3 -> 45.9, 12012 111 -> 101, 3121
    // (Rader) 148 -> 124; the longest one-pass convolutions lose (3851 187 -> 206).
    // Generic and four: 72 to 73, 57.3, 47.9, 102, 125, 207; eight: 72.3, 55.8, 47.4, 100,
    // 124, 210.  Radices above 16 run one wave per SIMD and are faster as they were (1023 x
    // 2000 80 us in this form, 77).
    constexpr bool TWG = sizeof(T) == 4 || !PRE || MAXE > 16;
    // staged at the start of the tile (FP64 only: the FP32 passes are faster with
    // the registers the second path would take, and prefetch instead)
    const bool tw_in_lds = sizeof(T) == 8 && A.tw_lds != 0;
    cx<T> w[NB][R - 1];
    if (early && !tw_in_lds && ns > 1) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const uint32_t b = lane + i * tpi;
            if (act && b < nb) {
                const cx<T>* tw = gmem<const cx<T>>(A.tw) + tw_off + mod_ns(b) * (R - 1);
#pragma unroll
                for (int r = 1; r < R; ++r)
                    w[i][r - 1] = tw[r - 1];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const uint32_t b = lane + i * tpi;
        if (act && b < nb) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                v[i][r] = my[lds_index<T>(b + r * nb)];
        } else if constexpr (MF) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                v[i][r] = {T(0), T(0)};
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const uint32_t b = lane + i * tpi;
        const bool ok = act && b < nb;
        const uint32_t k = (ns == 1) ? 0u : mod_ns(b);
        if (ok && ns > 1) {
            if (tw_in_lds) {
                const cx<T>* tw = ltw + tw_off + k * (R - 1);
#pragma unroll
                for (int r = 1; r < R; ++r)
                    v[i][r] = cmul(v[i][r], tw[r - 1]);
            } else {
                const cx<T>* tw =
                    (TWG ? gmem<const cx<T>>(A.tw) : (const cx<T>*)A.tw) + tw_off + k * (R - 1);
#pragma unroll
                for (int r = 1; r < R; ++r)
                    v[i][r] = cmul(v[i][r], early ? w[i][r - 1] : tw[r - 1]);
            }
        }
        if constexpr (MF)
            dft16_mfma<DK>(reinterpret_cast<cx<float>*>(v[i]), K); // the whole wave
        else if (ok)
            dft<T, R>(v[i]);
        if (ok) {
            const uint32_t base = (b - k) * R + k;
            if constexpr (IO == ST_OUT) {
                const KfaIo& io = A.out;
                const Ctx cio = make_ctx(io, inst);
                const int64_t es = (int64_t)io.e_mul * io.stride;
                const int64_t a0 = cio.base + (int64_t)cio.lgb * io.stride;
                const bool cj = ((io.flags & KFA_IO_CONJ1) != 0) != ((io.flags & KFA_IO_CONJ2) != 0);
                if (io.flags & KFA_IO_SCALE) {
                    const T sc = (T)A.scale;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        v[i][r].re *= sc;
                        v[i][r].im *= sc;
                    }
                }
                if (io.flags & KFA_IO_REAL) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        gmem<T>(io.ptr)[a0 + (int64_t)(base + r * ns) * es] = v[i][r].re;
                } else {
                    if (cj) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[i][r].im = -v[i][r].im;
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        gmem<cx<T>>(io.ptr)[a0 + (int64_t)(base + r * ns) * es] = v[i][r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    my[lds_index<T>(base + r * ns)] = v[i][r];
            }
        }
    }
    if constexpr (IO != ST_OUT)
        __syncthreads();
}

// Arguments, uniform per workgroup, read through the constant address space: every
// field is a scalar load that the compiler may keep or hoist.  (The ragged
// executor's arguments lie in device memory.  Read as ordinary memory each use is
// a vector load with a wait of its own, repeated after every store and barrier
// because those might alias it.)  Nothing in the launch may write there.
template <typename A>
__device__ __forceinline__ const A& const_args(uint64_t p) {
    typedef const __attribute__((address_space(4))) A* CP;
    return *(const A*)(CP)p;
}
// the operands of a function called by whole waves arrive in vector registers:
// uniform ones back to scalar registers, an LDS pointer back to its address space
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}
template <typename P>
__device__ __forceinline__ uint32_t lds_offset(const P* p) {
    typedef const __attribute__((address_space(3))) P* LP;
    return (uint32_t)(uintptr_t)(LP)p;
}
template <typename P>
__device__ __forceinline__ P* lds_at(uint32_t off) {
    typedef __attribute__((address_space(3))) P* LP;
    return (P*)(LP)off;
}

// A stage as a function of its own (registers allocated per radix): `args` as for
// const_args, LDS operands as offsets.
template <typename T, int R, int MAXE, int IO>
__device__ __attribute__((noinline)) void lds_stage_fn(uint64_t args, uint32_t s, uint32_t my,
                                                       uint32_t lane, bool act, uint32_t ltw,
                                                       uint64_t inst) {
    const KfaFftArgs& A = const_args<KfaFftArgs>(uniform64(args));
    lds_stage<T, R, MAXE, IO, DFT_VALU, 0, 0, false>(
        A, __builtin_amdgcn_readfirstlane(s), lds_at<cx<T>>(my), lane, act, lds_at<cx<T>>(ltw),
        MfmaConst<DFT_VALU>(), inst);
}

#define KFA_STAGE_CASE(R)                                                                         \
    case R:                                                                                       \
        if constexpr (R <= MAXE && SEP) {                                                         \
            if (sio == ST_OUT)                                                                    \
                lds_stage_fn<T, R, MAXE, ST_OUT>((uint64_t)&A, s, lds_offset(my), lane, act,      \
                                                 lds_offset(ltw), first + il);                    \
            else                                                                                  \
                lds_stage_fn<T, R, MAXE, ST_LDS>((uint64_t)&A, s, lds_offset(my), lane, act,      \
                                                 lds_offset(ltw), 0);                             \
        } else if constexpr (R <= MAXE) {                                                         \
            if (sio == ST_OUT)                                                                    \
                lds_stage<T, R, MAXE, ST_OUT, DK>(A, s, my, lane, act, ltw, K, first + il);       \
            else                                                                                  \
                lds_stage<T, R, MAXE, ST_LDS, DK>(A, s, my, lane, act, ltw, K);                   \
        }                                                                                         \
        break;

// The stages of a compiled length LC from stage SI on; the last one stores to
// memory when out_last (plain row layouts), else to LDS.
template <typename T, int MAXE, int DK, int LC, int SI>
__device__ __forceinline__ void ct_stages(const KfaFftArgs& A, cx<T>* my, uint32_t lane, bool act,
                                          const cx<T>* ltw, const MfmaConst<DK>& K,
                                          uint64_t inst, bool out_last) {
    using M = Mix<LC>;
    if constexpr (SI < M::S) {
        constexpr int R = M::R(SI);
        if constexpr (SI + 1 == M::S) {
            if (out_last)
                lds_stage<T, R, MAXE, ST_OUT, DK, LC, SI>(A, SI, my, lane, act, ltw, K, inst);
            else
                lds_stage<T, R, MAXE, ST_LDS, DK, LC, SI>(A, SI, my, lane, act, ltw, K);
        } else {
            lds_stage<T, R, MAXE, ST_LDS, DK, LC, SI>(A, SI, my, lane, act, ltw, K);
        }
        ct_stages<T, MAXE, DK, LC, SI + 1>(A, my, lane, act, ltw, K, inst, out_last);
    }
}

// One workgroup tile of a pass: instances [first, first + ipw).  The
// workgroup may be larger than tpi * ipw (threads beyond it idle); LDS must
// hold ipw * inst_stride elements, then tw_lds stage twiddles (FP64).  SEP: every
// stage is a call (lds_stage_fn); A then is a const_args reference.
template <typename T, int MAXE, int DK = DFT_VALU, int LC = 0, bool SEP = false>
__device__ __forceinline__ void fft_tile(const KfaFftArgs& A, uint64_t first, cx<T>* lds,
                                         uint32_t tid) {
    MfmaConst<DK> K;
    if constexpr (DK != DFT_VALU)
        K = mfma_dft16_const<DK>();
    const uint32_t nin =
        (uint32_t)((A.batch - first) < (uint64_t)A.ipw ? (A.batch - first) : (uint64_t)A.ipw);
    const uint32_t L = A.L;

    // 1. load.  Thread -> (instance, lane) as in the stages: lanes of one instance
    // on consecutive threads (rows), or instances on consecutive threads (in_jfast,
    // columns); each thread walks elements lane, lane + tpi, ...
    const uint32_t tpi = A.tpi, ipw = A.ipw;
    // elements a thread loads or stores at a time (FP64: as many as the radices up to 16
    // leave registers for, see lds_stage)
    constexpr int IOB = sizeof(T) == 8 && MAXE == 16 ? 6 : 8;
    // plain row layouts: the last stage writes to memory directly (one LDS sweep
    // and one barrier fewer); column layouts keep the cooperative store, whose
    // consecutive threads walk instances
    const bool fuse_out = !A.out_jfast && A.nstages >= 2 && fused_io_plain(A.out, KFA_IO_SCALE);
    {
        const uint32_t j = A.in_jfast ? tid % ipw : tid / tpi;
        const uint32_t ln = A.in_jfast ? tid / ipw : tid % tpi;
        if (ln < tpi && j < nin) {
            const KfaIo& io = A.in;
            const Ctx c = make_ctx(io, first + j);
            cx<T>* dst = lds + (size_t)j * A.inst_stride;
            for (uint32_t e0 = ln; e0 < L; e0 += IOB * tpi) {
                cx<T> v[IOB];
                uint32_t eb[IOB];
                bool ok[IOB];
#pragma unroll
                for (int i = 0; i < IOB; ++i) {
                    eb[i] = e0 + i * tpi;
                    ok[i] = eb[i] < L;
                }
                load_elems<T, IOB, 1>(io, c, v, eb, ok, 0);
#pragma unroll
                for (int i = 0; i < IOB; ++i)
                    if (ok[i])
                        dst[lds_index<T>(eb[i])] = v[i];
            }
        }
    }
    // the stage twiddles, when staged, behind the instances
    cx<T>* ltw = lds + (size_t)ipw * A.inst_stride;
    if (sizeof(T) == 8 && A.tw_lds) {
        const cx<T>* g = gmem<const cx<T>>(A.tw);
        for (uint32_t i = tid; i < A.tw_lds; i += blockDim.x)
            ltw[i] = g[i];
    }
    __syncthreads();

    // 2. radix stages; a convolution pass (mid_pw) runs them twice around a
    // pointwise product and conjugation of the first round's spectrum
    const uint32_t il = tid / A.tpi, lane = tid - il * A.tpi;
    const bool act = il < nin;
    cx<T>* my = lds + (size_t)(act ? il : 0) * A.inst_stride;
    const uint32_t rounds = A.mid_pw ? 2u : 1u;
    for (uint32_t round = 0; round < rounds; ++round) {
        if (round == 1) {
            if (act) {
                const uint64_t row = (first + il) % A.mid_rows;
                if (A.mid_dc && row == 0 && lane == 0)
                    gmem<cx<T>>(A.mid_dc)[(first + il) / A.mid_rows] = my[lds_index<T>(0)];
                const cx<T>* h = gmem<const cx<T>>(A.mid_pw) + row * L;
                // factors held at a time (517 x 8112 FP32 156.6 us with eight, 153.1 with
                // four; 523 x 8019 132.1 and 129.8, 527 x 7958 70.4 and 67.4)
                constexpr int MB = 4;
                for (uint32_t e0 = lane; e0 < L; e0 += MB * tpi) {
                    cx<T> w[MB];
#pragma unroll
                    for (int i = 0; i < MB; ++i) {
                        const uint32_t e = e0 + i * tpi;
                        w[i] = h[e < L ? e : 0u];
                    }
#pragma unroll
                    for (int i = 0; i < MB; ++i) {
                        const uint32_t e = e0 + i * tpi;
                        if (e < L) {
                            cx<T> v = cmul(my[lds_index<T>(e)], w[i]);
                            v.im = -v.im;
                            my[lds_index<T>(e)] = v;
                        }
                    }
                }
            }
            __syncthreads();
        }
        if constexpr (LC != 0) {
            ct_stages<T, MAXE, DK, LC, 0>(A, my, lane, act, ltw, K, first + il,
                                          fuse_out && round + 1 == rounds);
            continue;
        }
        for (uint32_t s = 0; s < A.nstages; ++s) {
            const int sio =
                (fuse_out && round + 1 == rounds && s + 1 == A.nstages) ? ST_OUT : ST_LDS;
            switch (A.st[s].radix) {
                KFA_STAGE_CASE(2)
                KFA_STAGE_CASE(3)
                KFA_STAGE_CASE(4)
                KFA_STAGE_CASE(5)
                KFA_STAGE_CASE(7)
                KFA_STAGE_CASE(8)
                KFA_STAGE_CASE(9)
                KFA_STAGE_CASE(11)
                KFA_STAGE_CASE(13)
                KFA_STAGE_CASE(16)
                KFA_STAGE_CASE(17)
                KFA_STAGE_CASE(19)
                KFA_STAGE_CASE(23)
                KFA_STAGE_CASE(29)
                KFA_STAGE_CASE(31)
            default:
                break;
            }
        }
    }

    // 3. store, thread mapping as the load's (out_jfast)
    if (!fuse_out) {
        const bool addx0 = (A.out.flags & KFA_IO_ADDX0) != 0;
        const uint32_t j = A.out_jfast ? tid % ipw : tid / tpi;
        const uint32_t ln = A.out_jfast ? tid / ipw : tid % tpi;
        if (ln < tpi && j < nin) {
            const Ctx c = make_ctx(A.out, first + j);
            const cx<T>* srcl = lds + (size_t)j * A.inst_stride;
            if (A.out.flags & KFA_IO_RPOST) {
                store_real_post<T>(A.out, c, srcl, L, ln, tpi);
            } else {
                const cx<T> x0 = addx0 ? load_aux<T>(A.out, c) : cx<T>{T(0), T(0)};
                for (uint32_t e0 = ln; e0 < L; e0 += IOB * tpi) {
                    cx<T> v[IOB];
                    uint32_t eb[IOB];
                    bool ok[IOB];
#pragma unroll
                    for (int i = 0; i < IOB; ++i) {
                        eb[i] = e0 + i * tpi;
                        ok[i] = eb[i] < L;
                        v[i] = srcl[lds_index<T>(ok[i] ? eb[i] : 0u)];
                    }
                    store_elems<T, IOB, 1>(A, c, v, eb, ok, 0, x0);
                }
            }
        }
    }
}

template <typename T, int MAXE, int DK = DFT_VALU, int LC = 0>
__global__ void __launch_bounds__(MAXE <= 16 ? 512 : 256) k_fft(const KfaFftArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    uint32_t tile = blockIdx.x;
    if (A.xcds > 1) {
        // XCD x = b mod n takes tiles [x q + min(x, r), ...): q = G / n, r = G mod n
        const uint32_t n = A.xcds, G = gridDim.x, q = G / n, r = G - q * n;
        const uint32_t x = tile % n, j = tile / n;
        tile = x * q + (x < r ? x : r) + j;
    }
    fft_tile<T, MAXE, DK, LC>(A, (uint64_t)tile * A.ipw, reinterpret_cast<cx<T>*>(kfa_smem),
                             threadIdx.x);
}

template <typename T, int MAXE, int DK = DFT_VALU, int LC = 0>
static hipError_t launch_fft_impl(const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s) {
    // set once per process; the initialisation of a function-local static is
    // thread-safe, so plans executed from several threads agree on it
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_fft<T, MAXE, DK, LC>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess)
            (void)hipGetLastError(); // do not leave the error for the next launch
        return e;
    }();
    if (attr != hipSuccess)
        return attr;
    const uint64_t groups = (a.batch + a.ipw - 1) / a.ipw;
    if (groups == 0)
        return hipSuccess;
    if (groups > 0x7fffffffull)
        return hipErrorInvalidValue;
    // the split forms' matrix instructions and lane swaps span whole waves: such
    // workgroups are rounded up to a multiple of 64 threads (the extra threads
    // hold no instance and feed zeros), so that no lane of a wave lies outside
    // the workgroup
    const uint32_t threads = DK != DFT_VALU ? (a.tpi * a.ipw + 63) / 64 * 64 : a.tpi * a.ipw;
    hipLaunchKernelGGL((k_fft<T, MAXE, DK, LC>), dim3((unsigned)groups), dim3(threads), lds_bytes,
                       s, a);
    return hipGetLastError();
}

// The general pass with the stage schedule of a compiled length LC, where the
// arguments describe exactly that schedule (radix cap 16, vector units):
// hipErrorNotSupported otherwise.
template <typename T, int LC>
static hipError_t launch_fft_ct(const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s) {
    using M = Mix<LC>;
    if (a.L != (uint32_t)LC || a.nstages != (uint32_t)M::S || a.tpi != (uint32_t)M::TPI)
        return hipErrorNotSupported;
    for (int i = 0; i < M::S; ++i)
        if (a.st[i].radix != (uint32_t)M::R(i))
            return hipErrorNotSupported;
    return launch_fft_impl<T, 16, DFT_VALU, LC>(a, lds_bytes, s);
}

} // namespace kfa
