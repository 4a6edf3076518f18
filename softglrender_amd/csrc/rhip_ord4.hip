/*
 * rhip_ord4.hip -- the ordered rasters' kernels for 4x multisampled targets.
 */
#include "rhip_ord.h"

namespace rhip {

template void launchOrdShade<4>(const DrawParams &, int, int, hipStream_t);
template void launchOrdRest<4>(const DrawParams &, int, int, hipStream_t);
template void launchOrdered<4>(const DrawParams &, int, int, int, hipStream_t);

}  // namespace rhip
