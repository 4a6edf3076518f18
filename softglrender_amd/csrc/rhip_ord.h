/*
 * rhip_ord.h -- launches of the ordered rasters' kernels, one specialisation
 * per shading model (instantiated by rhip_ord1.hip and rhip_ord4.hip).
 */
#pragma once
#include "rhip_kernels.h"
#include "rhip_launch.h"

namespace rhip {

template <int S>
void launchOrdShade(const DrawParams &P, int grid, int need_deriv, hipStream_t st) {
  switch (P.shading) {
    case RHS_SHADING_BASIC: RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA RHS_SHADING_BASIC>, grid, 256, st, P, need_deriv); break;
    case RHS_SHADING_BLINN_PHONG:
      RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA RHS_SHADING_BLINN_PHONG>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_BLINN_PHONG_DIR:
      RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA RHS_SHADING_BLINN_PHONG_DIR>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_PBR: RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA RHS_SHADING_PBR>, grid, 256, st, P, need_deriv); break;
    case RHS_SHADING_IBL_IRRADIANCE:
    case RHS_SHADING_IBL_PREFILTER:
      /* a workgroup takes 1 to 16 fragments; `grid` blocks of 256 lanes cover them one lane each */
      RHIP_LAUNCH(k_ord_shade_ibl<S>, std::min(grid * 256, 2 * kIblGroups), kIblTerms + 64, st, P, need_deriv);
      break;
    case RHS_SHADING_SKYBOX:
    case RHS_SHADING_FXAA: RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA kShadingEnv>, grid, 256, st, P, need_deriv); break;
    default: RHIP_LAUNCH(k_ord_shade<S RHIP_COMMA RHS_SHADING_VERTEX_COLOR>, grid, 256, st, P, need_deriv); break;
  }
}

template <int S>
void launchOrdRest(const DrawParams &P, int grid, int need_deriv, hipStream_t st) {
  switch (P.shading) {
    case RHS_SHADING_BASIC: RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA RHS_SHADING_BASIC>, grid, 256, st, P, need_deriv); break;
    case RHS_SHADING_BLINN_PHONG:
      RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA RHS_SHADING_BLINN_PHONG>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_BLINN_PHONG_DIR:
      RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA RHS_SHADING_BLINN_PHONG_DIR>, grid, 256, st, P, need_deriv);
      break;
    case RHS_SHADING_PBR: RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA RHS_SHADING_PBR>, grid, 256, st, P, need_deriv); break;
    case RHS_SHADING_SKYBOX:
    case RHS_SHADING_IBL_IRRADIANCE:
    case RHS_SHADING_IBL_PREFILTER:
    case RHS_SHADING_FXAA: RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA kShadingEnv>, grid, 256, st, P, need_deriv); break;
    default: RHIP_LAUNCH(k_ord_rest<S RHIP_COMMA RHS_SHADING_VERTEX_COLOR>, grid, 256, st, P, need_deriv); break;
  }
}

template <int S>
void launchOrdered(const DrawParams &P, int ntiles, int need_deriv, int flush_each, hipStream_t st) {
  switch (P.shading) {
    case RHS_SHADING_BASIC: {
#define K_ORD k_raster_ord<S, RHS_SHADING_BASIC>
      RHIP_LAUNCH(K_ORD, ntiles, 256, st, P, need_deriv, flush_each);
#undef K_ORD
      break;
    }
    case RHS_SHADING_BLINN_PHONG: {
#define K_ORD k_raster_ord<S, RHS_SHADING_BLINN_PHONG>
      RHIP_LAUNCH(K_ORD, ntiles, 256, st, P, need_deriv, flush_each);
#undef K_ORD
      break;
    }
    case RHS_SHADING_BLINN_PHONG_DIR: {
#define K_ORD k_raster_ord<S, RHS_SHADING_BLINN_PHONG_DIR>
      RHIP_LAUNCH(K_ORD, ntiles, 256, st, P, need_deriv, flush_each);
#undef K_ORD
      break;
    }
    case RHS_SHADING_PBR: {
#define K_ORD k_raster_ord<S, RHS_SHADING_PBR>
      RHIP_LAUNCH(K_ORD, ntiles, 256, st, P, need_deriv, flush_each);
#undef K_ORD
      break;
    }
    default: {
#define K_ORD k_raster_ord<S, RHS_SHADING_VERTEX_COLOR>
      RHIP_LAUNCH(K_ORD, ntiles, 256, st, P, need_deriv, flush_each);
#undef K_ORD
      break;
    }
  }
}

}  // namespace rhip
