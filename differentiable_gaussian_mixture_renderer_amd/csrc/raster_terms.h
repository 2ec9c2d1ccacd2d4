// SPDX-License-Identifier: GPL-3.0-or-later
// Scalar terms of the volumetric rasteriser, usable on the host as well: the
// CPU tests hold their rounding against double.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define DGMR_RASTER_FN __host__ __device__ __forceinline__
#else
#define DGMR_RASTER_FN inline
#endif

namespace dgmr {

// What a slot of mass m lets through.  The library's exponential: 2^(m log2 e)
// in the hardware's rounds the product, 3.5e-6 of the value at m = 40 (rms
// 8.5e-8 against 2.4e-8 over the masses of a frame), and the merges compare
// costs weighed with these.
DGMR_RASTER_FN float slot_transmittance(float m) { return expf(-m); }

} // namespace dgmr
