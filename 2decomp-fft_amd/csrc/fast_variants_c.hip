// fast_variants_c.hip -- registered specialised kernels, part 3 of 5:
// 320 / 576 / 800 / 960 / 1000 / 1152, the 1280 / 1536 / 2048-point columns, the short lengths and the persistent batch tiles.
#include "fast_impl.h"

namespace d2dhip {

// 960 = 8·8·15 over 64 rows a line: 2, 2 and 1 butterflies a lane with 6, 6
// and 0 % of the slots idle (16·12·5: 6, 37 and 0 %, 24 values a lane)
using R8_8_15 = RList<8, 8, 15>;

std::vector<FastVariant> fast_variants_c() {
  return {
    // and 320, 576, 800, 960, 1000, 1152 (FP32 columns of 576, 960 and 1000 points
    // run on the any-length kernels: 4.3 -> 4.6, 3.8 -> 4.2, 3.4 -> 3.9 TB/s)
    D2D_VARIANTS(double, 320, 8, 256, false, R8_8_5),
    D2D_VARIANTS(double, 320, 4, 128, true, R8_8_5),
    D2D_VARIANTS(double, 576, 8, 512, false, R16_9_4),
    D2D_VARIANTS(double, 576, 4, 256, false, R16_9_4),
    D2D_VARIANTS(double, 576, 4, 256, true, R16_9_4),
    D2D_SPLIT_C2C(double, 576, 8, 512, false, R16_9_4, 4),
    D2D_VARIANTS(double, 800, 8, 512, false, R16_10_5),
    D2D_VARIANTS(double, 800, 4, 256, false, R16_10_5),
    D2D_VARIANTS(double, 800, 4, 256, true, R16_10_5),
    D2D_SPLIT_C2C(double, 800, 8, 512, false, R16_10_5, 4),
    D2D_VARIANTS(double, 960, 8, 512, false, R16_12_5),
    D2D_VARIANTS(double, 960, 4, 256, false, R16_12_5),
    D2D_VARIANTS(double, 960, 2, 256, true, R16_12_5),
    D2D_VARIANTS(double, 960, 4, 256, true, R16_12_5),
    D2D_SPLIT_C2C(double, 960, 8, 1024, false, R16_12_5, 4),
    make_variant<double, 960, 8, 512, IO_C2C, false, R8_8_15, 1, 4>(
        "double n=960 tx=8 nt=512 c2c xs w4 r8815"),
    make_variant<double, 960, 8, 512, IO_C2C, false, R8_8_15>("double n=960 tx=8 nt=512 c2c r8815"),
    make_variant<double, 960, 4, 256, IO_R2C, true, R8_8_15>("double n=960 tx=4 nt=256 r2c r8815"),
    make_variant<double, 960, 4, 256, IO_C2R, true, R8_8_15>("double n=960 tx=4 nt=256 c2r r8815"),
    D2D_SPLIT_C2C(double, 1000, 8, 512, false, R10_10_10, 4),
    D2D_VARIANTS(double, 1000, 8, 512, false, R10_10_10),
    D2D_VARIANTS(double, 1000, 4, 256, false, R10_10_10),
    D2D_VARIANTS(double, 1000, 2, 256, true, R10_10_10),
    D2D_VARIANTS(double, 1000, 4, 256, true, R10_10_10),
    D2D_SPLIT_C2C(double, 1000, 8, 1024, false, R10_10_10, 4),
    D2D_VARIANTS(double, 1152, 8, 512, false, R16_9_8),
    D2D_VARIANTS(double, 1152, 4, 256, false, R16_9_8),
    D2D_VARIANTS(double, 1152, 4, 256, true, R16_9_8),
    D2D_VARIANTS(double, 1152, 2, 256, true, R16_9_8),
    D2D_SPLIT_C2C(double, 1152, 8, 1024, false, R16_9_8, 4),
    D2D_VARIANTS(float, 320, 16, 512, false, R8_8_5),
    D2D_VARIANTS(float, 320, 4, 128, true, R8_8_5),
    D2D_VARIANTS(float, 576, 4, 256, true, R16_9_4),
    D2D_VARIANTS(float, 800, 16, 512, false, R16_10_5),
    D2D_VARIANTS(float, 800, 4, 256, true, R16_10_5),
    D2D_VARIANTS(float, 960, 4, 256, true, R16_12_5),
    D2D_VARIANTS(float, 1000, 4, 256, true, R10_10_10),
    D2D_VARIANTS(float, 1152, 16, 512, false, R16_9_8),
    D2D_VARIANTS(float, 1152, 4, 256, true, R16_9_8),
    // 1280, 1536 and 2048 points (columns of 1280 run on the any-length kernels:
    // FP64 4.0-4.2 -> 4.4 TB/s, FP32 3.1-3.3 -> 3.6)
    D2D_VARIANTS(double, 1280, 2, 256, true, R16_16_5),
    D2D_SPLIT_C2C(double, 1536, 8, 1024, false, R16_16_6, 4),
    D2D_VARIANTS(double, 1536, 4, 256, false, R16_16_6),
    D2D_VARIANTS(double, 1536, 2, 256, true, R16_16_6),
    D2D_SPLIT_C2C(double, 1536, 8, 512, false, R16_16_6, 4),
    // (the split-exchange 8-column tile first: the default of plans too
    // large to tune, measured 30-31 ms against 39 ms per 2048^3 FP64 stage)
    D2D_SPLIT_C2C(double, 2048, 8, 1024, false, R16_16_8, 4),
    D2D_VARIANTS(double, 2048, 4, 512, false, R16_16_8),
    D2D_VARIANTS(float, 1280, 4, 256, true, R16_16_5),
    D2D_VARIANTS(float, 1536, 8, 512, false, R16_16_6),
    D2D_VARIANTS(float, 1536, 4, 256, true, R16_16_6),
    D2D_VARIANTS(float, 2048, 8, 512, false, R16_16_8),
    D2D_VARIANTS(float, 2048, 2, 256, true, R16_16_8),
    // short power-of-two lengths: 128-byte rows on strided axes
    D2D_VARIANTS(double, 256, 8, 128, false, R16_16),
    D2D_VARIANTS(double, 256, 4, 64, true, R16_16),
    D2D_VARIANTS(double, 256, 8, 128, true, R16_16),
    D2D_VARIANTS(double, 128, 8, 64, false, R16_8),
    D2D_VARIANTS(double, 128, 16, 128, false, R16_8),
    D2D_VARIANTS(double, 128, 8, 64, true, R16_8),
    D2D_VARIANTS(double, 64, 8, 64, false, R8_8),
    D2D_VARIANTS(double, 64, 16, 128, true, R8_8),
    D2D_VARIANTS(double, 32, 16, 64, false, R8_4),
    D2D_VARIANTS(double, 32, 32, 128, true, R8_4),
    D2D_VARIANTS(double, 48, 16, 64, false, R12_4),
    D2D_VARIANTS(double, 48, 16, 64, true, R12_4),
    D2D_VARIANTS(double, 80, 16, 64, false, R4_4_5),
    D2D_VARIANTS(double, 80, 16, 64, true, R4_4_5),
    D2D_VARIANTS(double, 96, 16, 64, false, R12_8),
    D2D_VARIANTS(double, 96, 16, 64, true, R12_8),
    D2D_VARIANTS(double, 160, 8, 64, false, R4_4_10),
    D2D_VARIANTS(double, 160, 16, 128, false, R4_4_10),
    D2D_VARIANTS(double, 160, 8, 64, true, R4_4_10),
    D2D_VARIANTS(double, 192, 8, 128, false, R4_4_12),
    D2D_VARIANTS(double, 192, 8, 64, false, R4_4_12),
    D2D_VARIANTS(double, 192, 4, 64, true, R4_4_12),
    D2D_VARIANTS(double, 192, 8, 64, true, R4_4_12),
    // tiles of the persistent batch kernel not registered above
    D2D_C2C(double, 192, 8, 128, true, R4_4_12),
    D2D_C2C(double, 160, 8, 128, false, R4_4_10),
    D2D_C2C(double, 160, 8, 128, true, R4_4_10),
    D2D_C2C(double, 128, 16, 128, true, R16_8),
    D2D_C2C(double, 96, 16, 128, false, R12_8),
    D2D_C2C(double, 96, 16, 128, true, R12_8),
    D2D_C2C(double, 80, 16, 128, false, R4_4_5),
    D2D_C2C(double, 80, 16, 128, true, R4_4_5),
    D2D_C2C(double, 64, 16, 128, false, R8_8),
    D2D_C2C(double, 48, 32, 128, false, R12_4),
    D2D_C2C(double, 48, 32, 128, true, R12_4),
    D2D_C2C(double, 32, 32, 128, false, R8_4),
    D2D_VARIANTS(float, 256, 16, 256, false, R16_16),
    D2D_VARIANTS(float, 256, 4, 64, true, R16_16),
    D2D_VARIANTS(float, 128, 16, 128, false, R16_8),
    D2D_VARIANTS(float, 128, 8, 64, true, R16_8),
    D2D_VARIANTS(float, 64, 16, 128, false, R8_8),
    D2D_VARIANTS(float, 64, 16, 128, true, R8_8),
  };
}

}  // namespace d2dhip
