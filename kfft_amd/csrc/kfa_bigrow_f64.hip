// Double-precision long one-pass rows (KFA_BIGROW_F64).
#include "kfa_bigrow_impl.h"
#include "kfa_kernels.h"

namespace kfa {
hipError_t launch_bigrow_f64(const KfaFftArgs& a, hipStream_t s) {
    switch (a.L) {
#define KFA_BIGROW_LAUNCH(N)                                                                       \
    case N:                                                                                        \
        return launch_bigrow_t<double, N>(a, s);
        KFA_BIGROW_F64(KFA_BIGROW_LAUNCH)
#undef KFA_BIGROW_LAUNCH
    default:
        return hipErrorNotSupported;
    }
}
} // namespace kfa
