/*
 * rhip_shade.hip -- launches of the two-phase raster's shading, one
 * specialisation per shading model.
 */
#include "rhip_kernels.h"
#include "rhip_launch.h"

namespace rhip {

template <int S>
void launchShade(const DrawParams &P, int grid, int need_deriv, hipStream_t st) {
  switch (P.shading) {
    case RHS_SHADING_BASIC: RHIP_LAUNCH(k_shade<S RHIP_COMMA RHS_SHADING_BASIC>, grid, 256, st, P, need_deriv); break;
    case RHS_SHADING_BLINN_PHONG:
      RHIP_LAUNCH(k_shade<S RHIP_COMMA RHS_SHADING_BLINN_PHONG>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_BLINN_PHONG_DIR:
      RHIP_LAUNCH(k_shade<S RHIP_COMMA RHS_SHADING_BLINN_PHONG_DIR>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_PBR: RHIP_LAUNCH(k_shade<S RHIP_COMMA RHS_SHADING_PBR>, grid, 256, st, P, need_deriv); break;
    default: RHIP_LAUNCH(k_shade<S RHIP_COMMA RHS_SHADING_VERTEX_COLOR>, grid, 256, st, P, need_deriv); break;
  }
}

template void launchShade<1>(const DrawParams &, int, int, hipStream_t);
template void launchShade<4>(const DrawParams &, int, int, hipStream_t);

}  // namespace rhip
