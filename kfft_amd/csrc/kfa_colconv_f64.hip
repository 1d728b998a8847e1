// Double-precision column convolutions (KFA_COLCONV_LENGTHS).
#include "kfa_colconv_impl.h"
#include "kfa_kernels.h"

namespace kfa {
hipError_t launch_colconv_f64(uint32_t L, const ColConvArgs& a, hipStream_t s) {
    switch (L) {
#define KFA_COLCONV_LAUNCH(N)                                                                      \
    case N:                                                                                        \
        return launch_colconv_t<double, N>(a, s);
        KFA_COLCONV_LENGTHS(KFA_COLCONV_LAUNCH)
#undef KFA_COLCONV_LAUNCH
    default:
        return hipErrorNotSupported;
    }
}
} // namespace kfa
