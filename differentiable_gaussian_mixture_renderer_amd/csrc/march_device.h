// SPDX-License-Identifier: GPL-3.0-or-later
// Device pieces of the volumetric ray marcher: the border walk over the sample
// sections (sections.h), the 1D restriction of a 3D Gaussian to a ray, the normal cdf and
// their adjoints.  References: src/dgmr/marching_steps.h:28-220,
// src/dgmr/math.h:412-468, src/dgmr/grad/math.h:529-620.
#pragma once

#include "device_grad.h"
#include "device_math.h"
#include "sections.h"

namespace dgmr {

// vol_marcher.h:59-67
constexpr int kSections = 16;      // n_large_steps: section-list capacity
constexpr int kBorders = 128;      // n_small_steps
constexpr int kBins = kBorders - 1;
constexpr int kStepsPerGaussian = 32;
constexpr float kRelevanceSigma = 3.f;
constexpr float kFilterSD = 0.55f;

// sample<n> (marching_steps.h:202-220) as a generator: border i+1 from border i
template <class S, int CAP>
struct BorderWalk {
    int cur;
    S prev;
    template <class L>
    __device__ __forceinline__ void begin(const L& sec)
    {
        cur = 0;
        prev = sec.size ? sec.data.start(0) : S(0);
    }
    template <class L>
    __device__ __forceinline__ S next(const L& sec)
    {
        if (sec.size == 0)
            return S(0);
        const S end = sec.data.end(cur);
        const S v = dmin(end, prev + sec.data.dt(cur));
        if (cur < sec.size - 1 && v == end)
            ++cur;
        prev = v;
        return v;
    }
};

template <class S>
struct Ray1d {
    S weight, centre, var;
};

template <class S>
__device__ __forceinline__ S dexp(S v);
template <>
__device__ __forceinline__ float dexp<float>(float v) { return expf(v); }
template <>
__device__ __forceinline__ double dexp<double>(double v) { return exp(v); }

template <class S>
__device__ __forceinline__ S derf(S v);
template <>
__device__ __forceinline__ float derf<float>(float v) { return erff(v); }
template <>
__device__ __forceinline__ double derf<double>(double v) { return erf(v); }

template <class S>
__device__ __forceinline__ S sym3_det(const S* A)
{
    return A[0] * (A[3] * A[5] - A[4] * A[4]) - A[1] * (A[1] * A[5] - A[4] * A[2]) + A[2] * (A[1] * A[4] - A[3] * A[2]);
}

// normalisation of the 3D Gaussian with inverse covariance A
template <class S>
__device__ __forceinline__ S ray_norm3(S detA) { return sqrt_rn(detA) / S(15.749609945722419); } // sqrt((2 pi)^3)

// restriction of N(mu, A^-1) to o + t d (stroke::gaussian::intersect_with_ray_inv_C
// as used at math.h:436): variance 1/(d^T A d), centre d^T A (mu - o) / (d^T A d),
// weight = integral of the normalised density along the ray.  m = mu - o and
// norm3 = ray_norm3(det A) do not depend on the ray.
template <class S>
__device__ __forceinline__ Ray1d<S> intersect_ray_pre(const S* mu, const S* A, const S* m, S norm3, const S* o, const S* d)
{
    const S Ad0 = (A[0] * d[0] + A[1] * d[1]) + A[2] * d[2];
    const S Ad1 = (A[1] * d[0] + A[3] * d[1]) + A[4] * d[2];
    const S Ad2 = (A[2] * d[0] + A[4] * d[1]) + A[5] * d[2];
    const S q = (d[0] * Ad0 + d[1] * Ad1) + d[2] * Ad2;
    const S C = S(1) / q;
    const S centre = ((Ad0 * m[0] + Ad1 * m[1]) + Ad2 * m[2]) * C;
    const S r0 = (o[0] + centre * d[0]) - mu[0];
    const S r1 = (o[1] + centre * d[1]) - mu[1];
    const S r2 = (o[2] + centre * d[2]) - mu[2];
    const S Ar0 = (A[0] * r0 + A[1] * r1) + A[2] * r2;
    const S Ar1 = (A[1] * r0 + A[3] * r1) + A[4] * r2;
    const S Ar2 = (A[2] * r0 + A[4] * r1) + A[5] * r2;
    const S E = (r0 * Ar0 + r1 * Ar1) + r2 * Ar2;
    const S norm1 = S(1) / sqrt_rn(S(2 * kPi) * C);
    return { norm3 / norm1 * dexp(S(-0.5) * E), centre, C };
}

template <class S>
__device__ __forceinline__ Ray1d<S> intersect_ray(const S* mu, const S* A, const S* o, const S* d)
{
    const S m[3] = { mu[0] - o[0], mu[1] - o[1], mu[2] - o[2] };
    return intersect_ray_pre(mu, A, m, ray_norm3(sym3_det(A)), o, d);
}

// the ray's nearest point (in the A-norm) to mu, minus mu, rounded as the
// restriction rounds it
template <class S>
__device__ __forceinline__ void ray_residual(const S* mu, const S* o, const S* d, S centre, S* r)
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
        r[i] = (o[i] + centre * d[i]) - mu[i];
}

// adjoint w.r.t. mu and the stored inverse covariance; g_wW is the gradient
// of the weight times the weight.  Gradient values only: contraction and (in
// float) hardware reciprocals.
template <class S>
__device__ __forceinline__ void intersect_ray_grad(const S* mu, const S* A, const S* o, const S* d, S centre, S g_wW, S g_centre, S g_var,
    S* g_mu, S* g_A)
{
#pragma clang fp contract(fast)
    S r[3];
    ray_residual(mu, o, d, centre, r);
    const S Ad[3] = { (A[0] * d[0] + A[1] * d[1]) + A[2] * d[2], (A[1] * d[0] + A[3] * d[1]) + A[4] * d[2],
        (A[2] * d[0] + A[4] * d[1]) + A[5] * d[2] };
    const S C = fast_div(S(1), dot3(d, Ad));
    const S Ar[3] = { (A[0] * r[0] + A[1] * r[1]) + A[2] * r[2], (A[1] * r[0] + A[3] * r[1]) + A[4] * r[2],
        (A[2] * r[0] + A[4] * r[1]) + A[5] * r[2] };
    const S gc = g_centre * C;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        g_mu[i] = g_wW * Ar[i] + gc * Ad[i];
    // A^-1 via the adjugate
    const S c00 = A[3] * A[5] - A[4] * A[4], c01 = A[2] * A[4] - A[1] * A[5], c02 = A[1] * A[4] - A[2] * A[3];
    const S inv_det = fast_div(S(1), (A[0] * c00 + A[1] * c01) + A[2] * c02);
    const S Ai[6] = { c00 * inv_det, c01 * inv_det, c02 * inv_det, (A[0] * A[5] - A[2] * A[2]) * inv_det, (A[2] * A[1] - A[0] * A[4]) * inv_det,
        (A[0] * A[3] - A[1] * A[1]) * inv_det };
    // g_A = g_wW / 2 (A^-1 - C d d^T - r r^T) - g_centre C / 2 (d r^T + r d^T) - g_var C^2 d d^T
    // (A^-1 - C d d^T is formed first: the two nearly cancel along the ray)
    const S h = S(0.5) * g_wW, f = g_var * (C * C), e = S(0.5) * gc;
    const int idx[6][2] = { { 0, 0 }, { 0, 1 }, { 0, 2 }, { 1, 1 }, { 1, 2 }, { 2, 2 } };
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int i = idx[k][0], j = idx[k][1];
        const S dd = d[i] * d[j];
        const S G = h * ((Ai[k] - C * dd) - r[i] * r[j]) - f * dd - e * (d[i] * r[j] + r[i] * d[j]);
        g_A[k] = (i == j) ? G : S(2) * G;
    }
}

// stroke::gaussian::cdf_inv_SD: standard normal cdf of (x - centre) / sd
template <class S>
__device__ __forceinline__ S cdf_inv_sd(S centre, S inv_sd, S x)
{
    return S(0.5) * (S(1) + derf((x - centre) * inv_sd * S(0.70710678118654752440)));
}

// The float path's cdf, the marcher's innermost operation (one per bin and
// Gaussian): erf by Abramowitz & Stegun, Handbook of Mathematical Functions,
// formula 7.1.26, erf(x) = 1 - t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) e^{-x^2}
// with t = 1 / (1 + p x), x >= 0, |error| <= 1.5e-7: one reciprocal and one
// exponential instead of a library erf.  The double path keeps erf.
// v: z / sqrt 2, e: e^{-v^2}
__device__ __forceinline__ float cdf_exp(float v, float* e)
{
    const float a = fabsf(v);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, a, 1.f));
    const float poly = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f), -0.284496736f), 0.254829592f);
    *e = __builtin_amdgcn_exp2f(-a * a * 1.4426950408889634f);
    return fmaf(0.5f, copysignf(fmaf(-poly, *e, 1.f), v), 0.5f);
}
template <>
__device__ __forceinline__ float cdf_inv_sd<float>(float centre, float inv_sd, float x)
{
    float e;
    return cdf_exp((x - centre) * inv_sd * 0.70710678118654752440f, &e);
}

// The cdf at x and what its derivatives need, for the adjoint of a bin's mass:
// p ~ pdf and q ~ z pdf up to the constant factors of cdf_grad_scale (d cdf /
// d centre = -inv_sd pdf, d cdf / d inv_sd = (x - centre) pdf).  Double: erf
// and exp.  Float: the cdf above, whose e^{-v^2} with v = z / sqrt 2 is the
// density's e^{-z^2 / 2}, so one exponential serves both.
__device__ __forceinline__ void cdf_grad_step(double centre, double inv_sd, double x, double* cdf, double* p, double* q)
{
    const double z = (x - centre) * inv_sd;
    *cdf = 0.5 * (1.0 + derf(z * 0.70710678118654752440));
    *p = dexp(-0.5 * z * z);
    *q = z * *p;
}
__device__ __forceinline__ void cdf_grad_step(float centre, float inv_sd, float x, float* cdf, float* p, float* q)
{
    const float v = (x - centre) * inv_sd * 0.70710678118654752440f;
    *cdf = cdf_exp(v, p);
    *q = v * *p;
}
// factors that turn sums over p into sums over inv_sd pdf, and over q into sums over z pdf
__device__ __forceinline__ void cdf_grad_scale(double inv_sd, double* fp, double* fq)
{
    *fp = inv_sd * 0.39894228040143267794;
    *fq = 0.39894228040143267794;
}
__device__ __forceinline__ void cdf_grad_scale(float inv_sd, float* fp, float* fq)
{
    *fp = inv_sd * 0.39894228040143267794f;
    *fq = 0.39894228040143267794f * 1.41421356237309504880f;
}

// pixel ray, vol_marcher_forward.cu:308-315
template <class S>
__device__ __forceinline__ void pixel_ray(const DevCamera<S>& cam, int px, int py, S* dir)
{
    const S pix0 = S(px) + S(0.5), pix1 = S(py) + S(0.5);
    const S ndc[3] = { pix0 * S(2) / S(cam.width) - S(1), pix1 * S(2) / S(cam.height) - S(1), S(0) };
    S v[4];
    transform_point(cam.inv_proj, ndc, v, 4);
    S p[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        p[i] = v[i] / v[3] - cam.pos[i];
    const S inv_len = S(1) / sqrt_rn(dot3(p, p));
#pragma unroll
    for (int i = 0; i < 3; ++i)
        dir[i] = p[i] * inv_len;
}

// ------------------------------------------------ windows along a tile's rays
// Where along any ray of the tile a staged Gaussian can matter: outside
// [lo, hi] it holds neither a sample section nor a bin mass of 1e-5.  One
// float pair per list entry, read by one lane each.
struct Reach1d {
    float lo, hi;
};

// the direction the tile's rays deviate from by at most dev
struct TileAxis {
    float dc[3];
    float dev;
};

// The part of a tile's rays near a Gaussian.  A point x d of a ray lies at
// A-distance^2 E + z^2 from the centre mu (E: of the ray's nearest point, z:
// standard deviations along the ray), so |x d - m| <= K sqrt(lambda) for every
// point with E + z^2 <= K^2, lambda the largest eigenvalue of A^-1 (bounded by
// the Frobenius norm), m = mu - o; as long as the rays point towards m that
// bounds x >= 0 by |m| +- K sqrt(lambda).  The mass on a ray is at most
// M exp(-E / 2) with M = mass norm3 sqrt(2 pi lambda).  Rounding is covered by
// a widened K and an absolute term; where it could not be (ill-conditioned A)
// and for rays that may point away from the Gaussian, bounded is false.
struct GaussianExtent {
    float len, sqrt_lam, err, mass; // |m|, sqrt(lambda), rounding, M
    bool bounded;
};

__device__ __forceinline__ GaussianExtent gaussian_extent(const float* A, float det, const float* m, float mass_norm3, const TileAxis& ax)
{
    GaussianExtent e { 0.f, 0.f, 0.f, 0.f, false };
    if (!(A[0] > 0.f && A[0] * A[3] - A[1] * A[1] > 0.f && det > 0.f))
        return e;
    const float id = 1.f / det;
    const float c0 = (A[3] * A[5] - A[4] * A[4]) * id, c1 = (A[2] * A[4] - A[1] * A[5]) * id, c2 = (A[1] * A[4] - A[2] * A[3]) * id,
                c3 = (A[0] * A[5] - A[2] * A[2]) * id, c4 = (A[2] * A[1] - A[0] * A[4]) * id, c5 = (A[0] * A[3] - A[1] * A[1]) * id;
    const float lam = sqrtf(c0 * c0 + c3 * c3 + c5 * c5 + 2.f * (c1 * c1 + c2 * c2 + c4 * c4));
    const float tr = A[0] + A[3] + A[5];
    const float cond = tr * lam;
    e.len = sqrtf(m[0] * m[0] + m[1] * m[1] + m[2] * m[2]);
    e.sqrt_lam = sqrtf(lam);
    e.err = 1e-6f * cond * e.len;
    e.mass = mass_norm3 * (2.5066282746310002f * e.sqrt_lam);
    e.bounded = cond < 1e4f && 1e-6f * e.len * sqrtf(tr) < 0.02f && e.mass == e.mass
        && m[0] * ax.dc[0] + m[1] * ax.dc[1] + m[2] * ax.dc[2] > 1.01f * ax.dev * e.len + 1e-6f * e.len;
    return e;
}

// half the window of the points with E + z^2 <= 2 ln M + above
__device__ __forceinline__ float extent_half(const GaussianExtent& e, float above)
{
    return (1.02f * sqrtf(fmaxf(2.f * logf(e.mass) + above, 0.f)) + 0.1f) * e.sqrt_lam + e.err;
}

// the block's common ray direction (its first pixel's) and the largest
// deviation of its pixels' rays from it
template <class S>
__device__ __forceinline__ TileAxis tile_axis(const S* d, bool inside, float* s_axis)
{
    if (threadIdx.x == 0) {
        // thread 0's pixel is inside in every tile
        s_axis[0] = float(d[0]);
        s_axis[1] = float(d[1]);
        s_axis[2] = float(d[2]);
        s_axis[3] = 0.f;
    }
    __syncthreads();
    TileAxis ax;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        ax.dc[k] = s_axis[k];
    const float e0 = float(d[0]) - ax.dc[0], e1 = float(d[1]) - ax.dc[1], e2 = float(d[2]) - ax.dc[2];
    const float dev = inside ? sqrtf(e0 * e0 + e1 * e1 + e2 * e2) : 0.f;
    atomicMax(reinterpret_cast<uint32_t*>(s_axis + 3), __float_as_uint(dev)); // dev >= 0: ordered as its bits
    __syncthreads();
    ax.dev = s_axis[3];
    return ax;
}

__device__ __forceinline__ uint64_t uniform_u64(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return (uint64_t(hi) << 32) | lo;
}

// the valid entries of a 64-entry word of a batch of cnt
__device__ __forceinline__ uint64_t valid_entries(int j0, int cnt)
{
    const int n = cnt - j0;
    return n >= 64 ? ~uint64_t(0) : ((uint64_t(1) << n) - 1);
}

// entries of a word whose window meets (wlo, whi): one entry per lane; none meets
// an empty window, also those without bounds
__device__ __forceinline__ uint64_t entries_in(const Reach1d* s_win, int j0, int cnt, float wlo, float whi)
{
    if (wlo > whi)
        return 0;
    const Reach1d w = s_win[min(j0 + int(lane_id()), cnt - 1)];
    return __builtin_amdgcn_ballot_w64(!(w.lo > whi) && !(w.hi < wlo)) & valid_entries(j0, cnt);
}

__device__ __forceinline__ float wave_min(float v)
{
#pragma unroll
    for (int k = 32; k > 0; k >>= 1)
        v = fminf(v, __shfl_xor(v, k));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

__device__ __forceinline__ float wave_max(float v) { return -wave_min(-v); }

template <int CTRL, int ROW_MASK = 0xf, int BANK_MASK = 0xf>
__device__ __forceinline__ double dpp_f64(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(b & 0xffffffffll), CTRL, ROW_MASK, BANK_MASK, true);
    const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, ROW_MASK, BANK_MASK, true);
    return __longlong_as_double((long long)(uint32_t(lo)) | ((long long)hi << 32));
}

__device__ __forceinline__ double wave_sum_to_last(double v)
{
    v += dpp_f64<0x111>(v);
    v += dpp_f64<0x112>(v);
    v += dpp_f64<0x114>(v);
    v += dpp_f64<0x118>(v);
    v += dpp_f64<0x142, 0xa>(v);
    v += dpp_f64<0x143, 0xc>(v);
    return v;
}

} // namespace dgmr
