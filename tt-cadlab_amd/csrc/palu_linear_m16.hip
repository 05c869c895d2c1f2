// The decode-step projections (palu_linear_kernel.h) for at most 16 rows.
#include "palu_linear_kernel.h"

namespace palu {

hipError_t linear_m16(int epi, int x_tiled, int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16,
                      int kt_total, int ks, int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep,
                      hipStream_t s) {
  return launch_mt<1>(epi, x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
}

}  // namespace palu
