// The 128-row tilings of the one-wave-per-SIMD prefill kernel (gemm_wide.h).
#include "gemm_wide.h"

namespace w4a16 {

hipError_t launch_wide_128x256(const GemmArgs& a, bool any, int split, float* part, int cus,
                               hipStream_t st) {
  return launch_wide_tiling<8, false, 4, 1, true>(a, any, split, part, cus, st);
}

hipError_t launch_wide_128x128(const GemmArgs& a, bool any, int split, float* part, int cus,
                               hipStream_t st) {
  return launch_wide_tiling<8, false, 2, 2, true>(a, any, split, part, cus, st);
}

}  // namespace w4a16
