/*
 * rhip_raster.hip -- launches of a single draw's two-phase raster.
 */
#include "rhip_kernels.h"
#include "rhip_launch.h"

namespace rhip {

/* Wavefronts per tile of a single draw's two-phase raster: four for 4x targets,
 * two without MSAA, whose tiles carry a quarter of the samples (measured on the
 * C2 frame: 2048^2 shadow pass 126 -> 111 us with two; the 4x pass 114 -> 152 us). */
template <int S>
constexpr int visWaves() {
  return S == 4 ? 4 : 2;
}

template <int S>
void launchHiz(const DrawParams &P, int ncoarse, hipStream_t st) {
  const int f = P.st.depthFunc;
  if (f == 4 || f == 6) {
    RHIP_LAUNCH(k_hiz_coarse<S RHIP_COMMA true>, ncoarse, 256, st, P);
  } else {
    RHIP_LAUNCH(k_hiz_coarse<S RHIP_COMMA false>, ncoarse, 256, st, P);
  }
}

template <int S>
void launchVis(const DrawParams &P, int ntiles, hipStream_t st) {
  const int f = P.st.depthFunc;
  switch (f) {
    case 1: RHIP_LAUNCH(k_raster_vis<S RHIP_COMMA VIS_LESS RHIP_COMMA kTile RHIP_COMMA visWaves<S>()>, ntiles, 64 * visWaves<S>(), st, P); break;
    case 3: RHIP_LAUNCH(k_raster_vis<S RHIP_COMMA VIS_LEQUAL RHIP_COMMA kTile RHIP_COMMA visWaves<S>()>, ntiles, 64 * visWaves<S>(), st, P); break;
    case 4: RHIP_LAUNCH(k_raster_vis<S RHIP_COMMA VIS_GREATER RHIP_COMMA kTile RHIP_COMMA visWaves<S>()>, ntiles, 64 * visWaves<S>(), st, P); break;
    default: RHIP_LAUNCH(k_raster_vis<S RHIP_COMMA VIS_GEQUAL RHIP_COMMA kTile RHIP_COMMA visWaves<S>()>, ntiles, 64 * visWaves<S>(), st, P); break;
  }
}

template void launchHiz<1>(const DrawParams &, int, hipStream_t);
template void launchHiz<4>(const DrawParams &, int, hipStream_t);
template void launchVis<1>(const DrawParams &, int, hipStream_t);
template void launchVis<4>(const DrawParams &, int, hipStream_t);

}  // namespace rhip
