// The 256-row tiling of the one-wave-per-SIMD prefill kernel (gemm_wide.h).
#include "gemm_wide.h"

namespace w4a16 {

hipError_t launch_wide_256(const GemmArgs& a, int split, float* part, int cus, hipStream_t st) {
  return launch_wide_tiling<16, true, 4, 1, false>(a, false, split, part, cus, st);
}

}  // namespace w4a16
