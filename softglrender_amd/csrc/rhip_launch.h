/*
 * rhip_launch.h -- launches of the draw kernels that live in translation units
 * of their own (they take most of the compile time): rhip_raster.hip,
 * rhip_shade.hip, rhip_ord1.hip and rhip_ord4.hip. S is the target's samples
 * per pixel (1 or 4).
 */
#pragma once
#include <hip/hip_runtime.h>

#include "rhip_internal.h"

/* Every kernel launch goes through this macro (one place to change how kernels are started). */
/* a comma inside a macro argument (template argument lists) */
#define RHIP_COMMA ,

#ifndef RHIP_LAUNCH
#define RHIP_LAUNCH(kern, grid, block, stream, ...) kern<<<(grid), (block), 0, (stream)>>>(__VA_ARGS__)
#endif

namespace rhip {

/* Two-phase raster: coarse hierarchical Z, then visibility and depth per tile. */
template <int S>
void launchHiz(const DrawParams &P, int ncoarse, hipStream_t st);
template <int S>
void launchVis(const DrawParams &P, int ntiles, hipStream_t st);
/* Shading of the fragments the two-phase raster queued. */
template <int S>
void launchShade(const DrawParams &P, int grid, int need_deriv, hipStream_t st);
/* Shading of the listed ordered raster's fragments, and its fallback for tiles that did not fit. */
template <int S>
void launchOrdShade(const DrawParams &P, int grid, int need_deriv, hipStream_t st);
template <int S>
void launchOrdRest(const DrawParams &P, int grid, int need_deriv, hipStream_t st);
/* Ordered raster (every state the two-phase raster does not take). */
template <int S>
void launchOrdered(const DrawParams &P, int ntiles, int need_deriv, int flush_each, hipStream_t st);

}  // namespace rhip
