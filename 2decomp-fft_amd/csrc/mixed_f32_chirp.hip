// mixed_f32_chirp.hip -- the FP32 kernels of lengths with a prime factor above 17
// (mixed_impl.h).
#include "mixed_impl.h"

namespace d2dhip {

std::vector<FastVariant> mixed_variants_f32_chirp() { return {D2D_MIXED_ALL(float, 2, " chirp")}; }

}  // namespace d2dhip
