// Single-precision shaped passes with the general fused IO (KFA_MIXGEN_LENGTHS).
#include "kfa_kernels.h"
#include "kfa_mixed_impl.h"

namespace kfa {
hipError_t launch_mixgen_f32(const KfaFftArgs& a, hipStream_t s) {
    switch (a.L) {
#define KFA_MIXGEN_LAUNCH(N)                                                                       \
    case N:                                                                                        \
        return launch_mixgen_t<float, N>(a, s);
        KFA_MIXGEN_LENGTHS(KFA_MIXGEN_LAUNCH)
        KFA_MIXGEN_LAUNCH(8192) // (one pass in FP32 only)
#undef KFA_MIXGEN_LAUNCH
    default:
        return hipErrorNotSupported;
    }
}
} // namespace kfa
