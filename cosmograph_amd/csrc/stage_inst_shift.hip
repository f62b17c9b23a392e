// Instantiations of the stage kernel for the fused steps of the shift build
// (MODE_SHIFT): LDS-DMA staging on the 4x4x16 tile, orders 2 (with and without
// the KO halo), 4 and 6, FP64 and split precision.  Grids and gauges they do
// not cover run the method sequence (cg_rk4_steps).
#include "bssn_stage_kernel.h"

namespace cg {
std::vector<StageVariant>& shift_variants() {
  static std::vector<StageVariant> v;
  return v;
}

#define CG_SHIFT1(TS, PREC, R, H, WPE, LA)                                                                    \
  static const bool CG_CAT(shift_, __COUNTER__) = [] {                                                        \
    shift_variants().push_back(StageVariant{PREC, 2 * R, H, 4, 4, 16, WPE, LA, false, nullptr, nullptr, nullptr, \
                                            CG_DMA_L(TS, TS, R, H, 4, 4, 16, WPE, LA, MODE_SHIFT),            \
                                            CG_DMA_I(TS, TS, R, H, 4, 4, 16, WPE, LA, MODE_SHIFT), nullptr}); \
    return true;                                                                                              \
  }();
#define CG_SHIFT(R, H)                   \
  CG_SHIFT1(double, 0, R, H, 2, false)   \
  CG_SHIFT1(double, 0, R, H, 2, true)    \
  CG_SHIFT1(float, 1, R, H, 3, false)    \
  CG_SHIFT1(float, 1, R, H, 3, true)
CG_SHIFT(1, 1)
CG_SHIFT(1, 2)
CG_SHIFT(2, 2)
CG_SHIFT(3, 3)
}  // namespace cg
