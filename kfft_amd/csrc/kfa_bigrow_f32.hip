// Single-precision long one-pass rows (KFA_BIGROW_F32).
#include "kfa_bigrow_impl.h"
#include "kfa_kernels.h"

namespace kfa {
hipError_t launch_bigrow_f32(const KfaFftArgs& a, hipStream_t s) {
    switch (a.L) {
#define KFA_BIGROW_LAUNCH(N)                                                                       \
    case N:                                                                                        \
        return launch_bigrow_t<float, N>(a, s);
        KFA_BIGROW_F32(KFA_BIGROW_LAUNCH)
#undef KFA_BIGROW_LAUNCH
    default:
        return hipErrorNotSupported;
    }
}
} // namespace kfa
