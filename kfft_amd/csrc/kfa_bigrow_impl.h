// Rows longer than the one-pass limit of the other forms (4096 points FP64, 8192
// FP32) in one pass: one instance per workgroup, the shaped stages of
// kfa_mixed_impl.h with every exchange in halves (real parts, then imaginary
// parts), so that a row needs half its size in LDS and two workgroups share a CU.
//
// Bound by HBM where the two-pass form of the same length moves every element
// twice.  Each row is one chain of load, exchanges and store: the second workgroup
// and the halves' short phases are what overlaps them (6561 x 2560 FP64: 222 us in two
// passes of 81 x 81, 160 here, 3.4 TB/s; what is left is its twelve barriers and the
// stage twiddles, as many bytes from L2 as the row itself).
#pragma once
#include "kfa_mixed_impl.h"

namespace kfa {

// waves per SIMD: what two workgroups need (the registers then are 512 / waves)
template <int L>
constexpr int bigrow_wpe() {
    return (2 * ((Mix<L>::TPI + 63) / 64) + 3) / 4;
}

template <typename T, int L>
__global__ void __launch_bounds__(Mix<L>::TPI)
    __attribute__((amdgpu_waves_per_eu(bigrow_wpe<L>()))) k_bigrow(const KfaFftArgs A) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    mixgen_tile<T, L, 1, true, KFA_USE_ROWS>(A, blockIdx.x, reinterpret_cast<cx<T>*>(kfa_smem),
                                             threadIdx.x);
}

template <typename T, int L>
static hipError_t launch_bigrow_t(const KfaFftArgs& a, hipStream_t s) {
    constexpr int PSH = sizeof(T) == 8 ? KFA_PAD_SHIFT_F64 : KFA_PAD_SHIFT_F32;
    constexpr uint32_t lds = (uint32_t)(((L + (L >> PSH)) | 1) * sizeof(T));
    static_assert(lds <= 80 * 1024 && Mix<L>::TPI <= 1024, "two workgroups per CU");
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_bigrow<T, L>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess)
            (void)hipGetLastError(); // do not leave the error for the next launch
        return e;
    }();
    if (attr != hipSuccess)
        return attr;
    if (a.L != (uint32_t)L || a.batch > 0x7fffffffull)
        return hipErrorInvalidValue;
    if (!a.batch)
        return hipSuccess;
    hipLaunchKernelGGL((k_bigrow<T, L>), dim3((unsigned)a.batch), dim3(Mix<L>::TPI), lds, s, a);
    return hipGetLastError();
}

} // namespace kfa
