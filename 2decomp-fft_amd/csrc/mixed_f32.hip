// mixed_f32.hip -- the FP32 kernels of any length with factors 2-17
// (mixed_impl.h).
#include "mixed_impl.h"

namespace d2dhip {

std::vector<FastVariant> mixed_variants_f32() {
  return {D2D_MIXED_ALL(float, 0, ""), D2D_MIXED_ALL(float, 1, " primes")};
}

}  // namespace d2dhip
