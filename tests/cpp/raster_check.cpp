// Host build of the rasteriser's scalar terms (raster_terms.h) for the CPU tests.
#include "../../differentiable_gaussian_mixture_renderer_amd/csrc/raster_terms.h"

extern "C" void transmittance_batch(int n, const float* m, float* out)
{
    for (int i = 0; i < n; ++i)
        out[i] = dgmr::slot_transmittance(m[i]);
}
