// mixed_f64.hip -- the FP64 kernels of any length with factors 2-17
// (mixed_impl.h).
#include "mixed_impl.h"

namespace d2dhip {

std::vector<FastVariant> mixed_variants_f64() {
  return {D2D_MIXED_ALL(double, 0, ""), D2D_MIXED_ALL(double, 1, " primes")};
}

}  // namespace d2dhip
