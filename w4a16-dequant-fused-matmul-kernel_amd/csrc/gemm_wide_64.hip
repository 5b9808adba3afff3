// The 64-row tilings of the one-wave-per-SIMD prefill kernel (gemm_wide.h), and
// what is common to all of them on the host.
#include "gemm_wide.h"

namespace w4a16 {

hipError_t launch_wide_256(const GemmArgs& a, int split, float* part, int cus, hipStream_t st);
hipError_t launch_wide_128x256(const GemmArgs& a, bool any, int split, float* part, int cus,
                               hipStream_t st);
hipError_t launch_wide_128x128(const GemmArgs& a, bool any, int split, float* part, int cus,
                               hipStream_t st);

int wide_split_panels(int K, int split, int slices) {
  const int panels = (K + kBK - 1) / kBK, unit = 4 * slices;
  const int per = split > 1 ? (panels + split - 1) / split : panels;
  return (per + unit - 1) / unit * unit;
}

hipError_t launch_wide(const GemmArgs& a, int cfg, bool any, int split, float* part, int cus,
                       hipStream_t st) {
  switch (cfg) {
    case kWide256x256: return any ? hipErrorInvalidValue : launch_wide_256(a, split, part, cus, st);
    case kWide128x256: return launch_wide_128x256(a, any, split, part, cus, st);
    case kWide128x128: return launch_wide_128x128(a, any, split, part, cus, st);
    case kWide64x128: return launch_wide_tiling<4, false, 2, 2, true>(a, any, split, part, cus, st);
    case kWide64x64: return launch_wide_tiling<4, false, 1, 4, true>(a, any, split, part, cus, st);
    case kWide32x64: return launch_wide_tiling<2, false, 1, 4, false>(a, any, split, part, cus, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace w4a16
