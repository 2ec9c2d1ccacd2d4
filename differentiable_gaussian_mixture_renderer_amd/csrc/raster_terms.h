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

// e^{-d^2 / (2 var)} for the borders of one Gaussian.  As 2^(d^2 scale) with the
// scale -log2(e) / (2 var) rounded once it is off by 4.4e-7 rms (the roundings
// of the scale and the product, times the exponent), where expf(-d^2 / 2 / var)
// is off by 2.9e-7; with the scale and the product in two parts, five
// instructions a border, by 2.1e-7.
struct DensityScale {
    float hi, lo; // their sum is -log2(e) / (2 var)
};

DGMR_RASTER_FN DensityScale density_scale(float var)
{
    constexpr float kHi = -0.72134752044448170f, kLo = -9.6298150e-9f; // -log2(e) / 2
#if defined(__HIP_DEVICE_COMPILE__)
    const float r = __builtin_amdgcn_rcpf(var);
#else
    const float r = 1.f / var;
#endif
    const float hi = kHi * r;
    return { hi, fmaf(kHi, r, -hi) + fmaf(fmaf(-var, r, 1.f), hi, kLo * r) };
}

DGMR_RASTER_FN float border_density(const DensityScale& s, float d)
{
    const float d2 = d * d;
    const float t = d2 * s.hi;
    // bounded: infinite once t or d2 is, where e is 0
    const float rest = fminf(fmaxf(fmaf(d2, s.lo, fmaf(d2, s.hi, -t)), -1.f), 1.f);
#if defined(__HIP_DEVICE_COMPILE__)
    const float e = __builtin_amdgcn_exp2f(t);
#else
    const float e = exp2f(t);
#endif
    return fmaf(e * 0.69314718055994531f, rest, e);
}

} // namespace dgmr
