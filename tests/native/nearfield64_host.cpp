// Host build of the FP64 near-field weight (hfmm0_amd/csrc/p2p_math.h), the same source the
// GPU kernels include, exported over arrays for tests/test_nearfield_fp64.py.
#include "../../hfmm0_amd/csrc/p2p_math.h"

using namespace hfmm::nearfield;

extern "C" {
void nf64_rsqrt(const double* r2, int n, double* rinv, double* r) {
    for (int i = 0; i < n; ++i) rsqrt64(r2[i], rinv[i], r[i]);
}
void nf64_sincospi(const double* y, int n, double* s, double* c) {
    for (int i = 0; i < n; ++i) sincospi_half64(y[i], SinCosPi64::pinned(), s[i], c[i]);
}
void nf64_weight(const double* r2, int n, double fl2, double k, double* wr, double* wi) {
    const HalfTurnK kp = halfturn_k(k);
    for (int i = 0; i < n; ++i) pair_weight64(r2[i], fl2, kp, SinCosPi64::pinned(), wr[i], wi[i]);
}
}
