// mixed_f64_chirp.hip -- the FP64 kernels of lengths with a prime factor above 17
// (mixed_impl.h).
#include "mixed_impl.h"

namespace d2dhip {

std::vector<FastVariant> mixed_variants_f64_chirp() { return {D2D_MIXED_ALL(double, 2, " chirp")}; }

}  // namespace d2dhip
