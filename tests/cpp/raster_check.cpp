// Host build of the rasteriser's scalar terms (raster_terms.h) for the CPU tests.
#include "../../differentiable_gaussian_mixture_renderer_amd/csrc/raster_terms.h"

extern "C" void transmittance_batch(int n, const float* m, float* out)
{
    for (int i = 0; i < n; ++i)
        out[i] = dgmr::slot_transmittance(m[i]);
}

extern "C" void density_batch(int n, const float* d, const float* var, float* out, float* plain)
{
    for (int i = 0; i < n; ++i) {
        out[i] = dgmr::border_density(dgmr::density_scale(var[i]), d[i]);
        plain[i] = expf(-0.5f * d[i] * d[i] / var[i]);
    }
}
