// Column convolution of two spectra in one pass: for every column x of two
// row-major matrices a and b (L rows), b = scale * conj(DFT(conj(DFT(a) DFT(b)))),
// the inverse transform of the product.  Both forward transforms, the product and
// the inverse run in one workgroup's LDS, on the schedule of the mixed-radix
// shaped passes (Mix<L>; the plan's stage twiddles): every element is read once
// and written once, 3 values of traffic per element against 7 for one-pass columns
// and 15 for two-pass ones (columns of a, of b, the product, columns back).
//
// Bound by latency: a tile holds 2 columns of 4160 rows (70 KB FP32), and one tile's
// ten waves share a CU, waiting 39% of their time for data and 34% to issue.  A row's
// access is 16 bytes of a 128-byte line; consecutive tiles take consecutive columns and
// run on one XCD, whose L2 then serves the line's other columns, and in blocks of four
// columns a line also holds the next three rows (5.9 million L2 requests in 140 us, a
// sixth of what its channels take).
// Measured, all columns of a real 4160 x 4160 convolution FP32 (2081 columns):
// 228 us as two-pass transforms and a product sweep, 190 in this pass on rows of
// the matrix, 138 on blocks; held to 96 registers for two workgroups per CU it
// spills (227).  FP64 without twiddle prefetch (372 bytes of spills with): the
// whole convolution 709 -> 599 us.
#pragma once
#include "kfa_mixed_impl.h"

namespace kfa {

// waves per SIMD that the LDS lets in (two tiles per CU where they fit)
template <typename T, int L, int IPW>
constexpr int colconv_wpe() {
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int lds = IPW * (int)sizeof(cx<T>) * ((L + (L >> PSH)) | 1);
    constexpr int waves = (IPW * Mix<L>::TPI + 63) / 64 * (2 * lds <= 160 * 1024 ? 2 : 1);
    return (waves + 3) / 4;
}

template <typename T, int L, int IPW>
__device__ __forceinline__ void colconv_tile(const ColConvArgs& A, uint64_t first, cx<T>* lds) {
    using M = Mix<L>;
    static_assert(M::valid() && M::S > 1, "length outside the mixed-radix passes");
    constexpr int E = M::E, TPI = M::TPI, NST = M::S;
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int SP = (L + (L >> PSH)) | 1;
    constexpr int R0 = M::R(0), NB0 = M::NB(0), STR0 = L / R0;
    constexpr int RL = M::R(NST - 1), NBL = M::NB(NST - 1), STRL = L / RL;
    // with registers for them: stage twiddles requested before the stage's barrier,
    // b's elements with a's
    constexpr bool PRE = sizeof(T) == 4 || colconv_wpe<T, L, IPW>() <= 2, early = sizeof(T) == 4;
    const uint32_t li = threadIdx.x % IPW, ll = threadIdx.x / IPW;
    const uint64_t col = first + li;
    const bool act = col < A.cols;
    // (threads past the last column read the tile's first one and store nothing)
    const uint64_t cr = act ? col : first;
    const uint64_t off = A.blk ? (cr >> 2) * A.blk + (cr & 3u) : cr;
    const int64_t pitch = A.blk ? 4 : (int64_t)A.pitch;
    cx<T>* my = lds + (size_t)li * SP;

    auto load = [&](const cx<T>* p, cx<T>* v) {
#pragma unroll
        for (int i = 0; i < NB0; ++i) {
            const int b = (int)ll + i * TPI;
#pragma unroll
            for (int r = 0; r < R0; ++r)
                v[i * R0 + r] = b < STR0 ? p[(int64_t)(b + r * STR0) * pitch] : cx<T>{T(0), T(0)};
        }
    };
    // stage 0 from registers, the others through LDS; outputs e = b + r STRL
    auto forward = [&](cx<T>* v) {
#pragma unroll
        for (int i = 0; i < NB0; ++i)
            dft<T, R0>(v + i * R0);
#pragma unroll
        for (int i = 0; i < NB0; ++i) {
            const int b = (int)ll + i * TPI;
            if (b < STR0) {
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    const int e = b * R0 + r;
                    my[e + (e >> PSH)] = v[i * R0 + r];
                }
            }
        }
        mixed_stages<T, L, 1, PRE>((const cx<T>*)A.tw, v, my, ll);
    };

    cx<T> va[E], v[E];
    load((const cx<T>*)A.a + off, va);
    if constexpr (early)
        load((const cx<T>*)A.b + off, v);
    forward(va);
    if constexpr (!early)
        load((const cx<T>*)A.b + off, v);
    __syncthreads(); // the last stage's LDS reads are done
    forward(v);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NBL; ++i) {
        const int b = (int)ll + i * TPI;
        if (b < STRL) {
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const int e = b + r * STRL;
                const cx<T> x = cmul(v[i * RL + r], va[i * RL + r]);
                my[e + (e >> PSH)] = {x.re, -x.im};
            }
        }
    }
    mixed_stages<T, L, 0, PRE>((const cx<T>*)A.tw, v, my, ll);
    if (act) {
        cx<T>* q = (cx<T>*)A.b + off;
        const T sc = (T)A.scale;
#pragma unroll
        for (int i = 0; i < NBL; ++i) {
            const int b = (int)ll + i * TPI;
            if (b < STRL) {
#pragma unroll
                for (int r = 0; r < RL; ++r)
                    q[(int64_t)(b + r * STRL) * pitch] = {v[i * RL + r].re * sc,
                                                          -(v[i * RL + r].im * sc)};
            }
        }
    }
}

// columns per tile: the largest power of two within 768 threads and 80 KB of LDS
// (two tiles per CU), two columns where those need up to 150 KB
template <typename T, int L>
constexpr int colconv_ipw() {
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr int bytes = (int)sizeof(cx<T>) * ((L + (L >> PSH)) | 1), TPI = Mix<L>::TPI;
    for (int ipw = 16; ipw > 1; ipw /= 2)
        if (ipw * TPI <= 768 && ipw * bytes <= (ipw == 2 ? 150 : 80) * 1024)
            return ipw;
    return 1;
}

template <typename T, int L, int IPW>
__global__ void __launch_bounds__(IPW* Mix<L>::TPI)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? colconv_wpe<T, L, IPW>() : 1))) k_colconv(const ColConvArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    uint32_t tile = blockIdx.x;
    if (A.xcds > 1) {
        const uint32_t n = A.xcds, G = gridDim.x, q = G / n, r = G - q * n;
        const uint32_t x = tile % n, j = tile / n;
        tile = x * q + (x < r ? x : r) + j;
    }
    colconv_tile<T, L, IPW>(A, (uint64_t)tile * IPW, reinterpret_cast<cx<T>*>(kfa_smem));
}

template <typename T, int L>
static hipError_t launch_colconv_t(const ColConvArgs& a, hipStream_t s) {
    constexpr int IPW = colconv_ipw<T, L>();
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr uint32_t lds = (uint32_t)(IPW * sizeof(cx<T>) * ((L + (L >> PSH)) | 1));
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_colconv<T, L, IPW>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess)
            (void)hipGetLastError(); // do not leave the error for the next launch
        return e;
    }();
    if (attr != hipSuccess)
        return attr;
    const uint64_t groups = (a.cols + IPW - 1) / IPW;
    if (!groups)
        return hipSuccess;
    if (groups > 0x7fffffffull)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_colconv<T, L, IPW>), dim3((unsigned)groups), dim3(IPW * Mix<L>::TPI),
                       lds, s, a);
    return hipGetLastError();
}

} // namespace kfa
