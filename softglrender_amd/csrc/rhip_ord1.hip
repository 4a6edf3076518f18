/*
 * rhip_ord1.hip -- the ordered rasters' kernels for single-sample targets.
 */
#include "rhip_ord.h"

namespace rhip {

template void launchOrdShade<1>(const DrawParams &, int, int, hipStream_t);
template void launchOrdRest<1>(const DrawParams &, int, int, hipStream_t);
template void launchOrdered<1>(const DrawParams &, int, int, int, hipStream_t);

}  // namespace rhip
