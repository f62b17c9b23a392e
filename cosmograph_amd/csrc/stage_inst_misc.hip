// Instantiations of the stage kernel: orders 2 and 8 (with and without the
// wider Kreiss-Oliger halo), both precisions: tiles with LDS-DMA twins, and the
// register-staged 4x8x8 tile for the grids that those do not fit.
#include "bssn_stage_kernel.h"

namespace cg {
std::vector<StageVariant>& stage_variants() {
  static std::vector<StageVariant> v;
  return v;
}

#define CG_MISC(R, H)                                                     \
  CG_REGISTER_STAGE(double, double, 0, R, H, 4, 8, 8, 1, true)             \
  CG_REGISTER_STAGE(double, double, 0, R, H, 4, 8, 8, 1, false)            \
  CG_REGISTER_STAGE(float, float, 1, R, H, 4, 8, 8, 1, true)               \
  CG_REGISTER_STAGE(float, float, 1, R, H, 4, 8, 8, 1, false)
// with LDS-DMA twins, at 2 (FP64) and W32 waves per SIMD
#define CG_MISC_D(R, H, TI, TJ, TK, W32)                                    \
  CG_REGISTER_STAGE_D(double, double, 0, R, H, TI, TJ, TK, 2, true)         \
  CG_REGISTER_STAGE_D(double, double, 0, R, H, TI, TJ, TK, 2, false)        \
  CG_REGISTER_STAGE_D(float, float, 1, R, H, TI, TJ, TK, W32, true)         \
  CG_REGISTER_STAGE_D(float, float, 1, R, H, TI, TJ, TK, W32, false)
CG_MISC_D(1, 1, 4, 4, 16, 3)
CG_MISC_D(1, 2, 4, 4, 16, 3)
CG_MISC_D(4, 4, 4, 4, 16, 2)
// 512 points: with a halo of 4 or 5 the FP64 tiles of 256 points fill the
// LDS of a CU with 4 waves (register staging; the DMA path at halo 5), this
// one with 8 at twice the LDS and a smaller halo share
CG_MISC_D(4, 4, 8, 8, 8, 2)
CG_MISC_D(4, 5, 8, 8, 8, 2)
CG_MISC(1, 1)
CG_MISC(1, 2)
CG_MISC(4, 4)
CG_MISC(4, 5)
}  // namespace cg
