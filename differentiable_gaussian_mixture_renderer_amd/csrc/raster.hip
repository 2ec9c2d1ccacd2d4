// SPDX-License-Identifier: GPL-3.0-or-later
// Volumetric rasteriser for gfx950 (reference: src/dgmr/vol_raster_forward.cu:36-520),
// forward only, as the reference.
//
//   1. k_splat_preprocess (the splatter's: cull, rect, tiles, xy, depth, SH
//      colour; the reference's preprocess computes the same quantities the
//      same way) and k_raster_extra: inverse of the filtered 3D covariance and
//      the filtered Ots mass per visible Gaussian.
//   2. bin_gaussians: the splatter's binning (same keys, same order).
//   3. k_raster_render: one 16x16 tile per 256-thread workgroup, one pixel per
//      thread.  Pass 1 sizes 32 bins per pixel (math::RasterBinSizer, kept in
//      registers, every slot indexed by a constant); pass 2 rasterises the
//      tile's Gaussians into the bins kChunk bins at a time and integrates each
//      chunk's bins piecewise-linearly before the next chunk, so only kChunk
//      bins of (rgb*mass, mass) and kChunk + 1 border evaluations are live.
#include <cmath>

#include "device_grad.h"
#include "device_math.h"
#include "host_common.h"
#include "march_device.h"
#include "raster_terms.h"
#include "splat_device.h"

namespace dgmr {
namespace {

constexpr int kRasterBins = 32;         // vol_raster::config::n_rasterisation_bins
constexpr int kRasterSteps = 256;       // vol_raster::config::n_steps_per_bin
constexpr float kRasterFilterSD = 0.55f; // vol_raster::config::filter_kernel_SD
constexpr float kRelevanceSigma = 3.f;  // vol_raster::config::gaussian_relevance_sigma
constexpr int kTile = 16;               // render_block_width/height (constants.h:45-46)
constexpr int kThreads = kTile * kTile;
constexpr int kChunk = 16;              // bins rasterised per walk of the tile's list
constexpr int kGroup = 4;               // bins evaluated together when some pixel of the wave needs one
constexpr int kBorderStride = kRasterBins + 1; // odd: one LDS row per pixel, conflict-free

// vol_raster_forward.cu:100-136 for the Gaussians the splatter preprocess kept:
// filtered inverse covariance (xx, xy, xz, yy, yz, zz) and the mass
// weight_to_mass<Ots>(w, scales + f^2, .) = w * 2 pi * (two largest of s + f^2)
__global__ __launch_bounds__(256) void k_raster_extra(int64_t n, SplatParams p, DevCamera<float> cam, const uint32_t* __restrict__ tiles,
    float* __restrict__ inv_cov, float* __restrict__ mass)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n || tiles[i] == 0)
        return;
    float s[3], q[4], w;
    gaussian_params(p, i, s, q, &w);
    const float mu[3] = { p.means[3 * i], p.means[3 * i + 1], p.means[3 * i + 2] };
    float cov[6];
    compute_cov(s, q, cov);
    const float dv[3] = { mu[0] - cam.pos[0], mu[1] - cam.pos[1], mu[2] - cam.pos[2] };
    const float aa = (kRasterFilterSD * cam.tan_fovx * 2.f) / float(cam.width);
    const float f = length3(dv) * aa;
    const float f2 = f * f;
    const float sf[3] = { s[0] + f2, s[1] + f2, s[2] + f2 };
    float la, lb;
    int i0, i1;
    larger2_values(sf, &la, &lb, &i0, &i1);
    mass[i] = w * (float(2 * kPi) * la * lb);
    const float cov_f[6] = { cov[0] + f2, cov[1], cov[2], cov[3] + f2, cov[4], cov[5] + f2 };
    float inv[6];
    sym3_inverse(cov_f, inv);
#pragma unroll
    for (int k = 0; k < 6; ++k)
        inv_cov[6 * i + k] = inv[k];
}

__device__ __forceinline__ float larger_of(float a, float b) { return a < b ? b : a; } // std::max(a, b)

// stroke::gaussian::integrate_normalised_SD over [a, b]
__device__ __forceinline__ float integrate_normalised_sd(float centre, float sd, float a, float b)
{
    const float k = 0.70710678118654752440f;
    return 0.5f * erff((b - centre) / sd * k) - 0.5f * erff((a - centre) / sd * k);
}

__device__ __forceinline__ float cdf_sd(float centre, float inv_sd, float x)
{
    return 0.5f * (1.f + erff((x - centre) * inv_sd * 0.70710678118654752440f));
}

// math::RasterBinSizer<vol_raster::config> (raster_bin_sizers.h:271-485)
struct BinSizer {
    float m[kRasterBins], b[kRasterBins], s[kRasterBins];
    float acc, maxd;

    __device__ __forceinline__ void init()
    {
#pragma unroll
        for (int i = 0; i < kRasterBins; ++i) {
            m[i] = 0.f;
            b[i] = __builtin_inff();
            s[i] = 0.f;
        }
        acc = 0.f;
        maxd = 0.f;
    }

    __device__ __forceinline__ void add(float mass, float centre, float sd)
    {
        if (mass < 0.0001f)
            return;
        constexpr int L = kRasterBins - 1;
        const float t_rel = centre + sd * kRelevanceSigma;
        const float added = mass * integrate_normalised_sd(centre, sd, 0.f, t_rel);
        maxd = larger_of(t_rel, maxd);
        acc += added;
        m[L] = added;
        b[L] = centre;
        s[L] = sd;
        // insertion from the back: swap while the left neighbour lies further
        bool moving = true;
        static_for<L>([&](auto q) {
            constexpr int i = L - q;
            const bool sw = moving && b[i - 1] > b[i];
            const float bl = b[i - 1], br = b[i], sl = s[i - 1], sr = s[i], ml = m[i - 1], mr = m[i];
            b[i - 1] = sw ? br : bl;
            b[i] = sw ? bl : br;
            s[i - 1] = sw ? sr : sl;
            s[i] = sw ? sl : sr;
            m[i - 1] = sw ? mr : ml;
            m[i] = sw ? ml : mr;
            moving = sw;
        });
        if (!(m[L] > 0.f))
            return;
        // every slot is taken: merge the cheapest adjacent pair
        float tr[L];
        float t = 1.f;
        static_for<L>([&](auto i) {
            t *= slot_transmittance(m[i]);
            tr[i] = t;
        });
        int best = -1;
        float best_val = __builtin_inff();
        static_for<L>([&](auto j) {
            float ta = 1.f;
            if constexpr (j > 0)
                ta = tr[j - 1];
            const float v = tr[j] * merge_cost(ta, tr[j], m[j], m[j + 1], b[j], b[j + 1], s[j], s[j + 1]);
            if (v < best_val) {
                best_val = v;
                best = j;
            }
        });
        // the reference asserts a candidate exists; with none its merge would
        // index slot -1, here slot 0 merges
        best = best < 0 ? 0 : best;
        // gather the pair (best, best + 1) without a runtime index
        float ba = b[0], bb = b[1], sa = s[0], sb = s[1], ma = m[0], mb = m[1], tb_a = 1.f, tb_b = tr[0];
        static_for<L - 1>([&](auto q) {
            constexpr int j = q + 1;
            const bool h = best == j;
            ba = h ? b[j] : ba;
            bb = h ? b[j + 1] : bb;
            sa = h ? s[j] : sa;
            sb = h ? s[j + 1] : sb;
            ma = h ? m[j] : ma;
            mb = h ? m[j + 1] : mb;
            tb_a = h ? tr[j - 1] : tb_a;
            tb_b = h ? tr[j] : tb_b;
        });
        float nm, nc, nsd;
        merge_values(tb_a, tb_b, ma, mb, ba, bb, sa, sb, &nm, &nc, &nsd);
        static_for<L>([&](auto j) {
            const bool here = j == best, after = j > best;
            b[j] = here ? nc : (after ? b[j + 1] : b[j]);
            s[j] = here ? nsd : (after ? s[j + 1] : s[j]);
            m[j] = here ? nm : (after ? m[j + 1] : m[j]);
        });
    }

    // kl(a, merged) + kl(b, merged) of two adjacent slots and their merge, kl of
    // normals (c1, s1), (c2, s2) being ((c1 - c2)^2 + s1^2 - s2^2) / (2 s2^2) +
    // log(s2 / s1): both logarithms as one, no square root (only variances are
    // needed), and the hardware reciprocal.  A merge computes 31 of these, which
    // was two thirds of pass 1's instructions as five divisions, two logarithms
    // and a square root each; its relative error against double is 5.8e-6 rms over
    // the pairs of a frame where that form's is 6.6e-6.  A Gaussian behind the camera
    // adds a negative mass, and a pair of one may merge to a negative variance:
    // the ratio is then negative and the cost NaN, which is never the cheapest.
    static __device__ __forceinline__ float merge_cost(float tb_a, float tb_b, float ma, float mb, float ba, float bb, float sa, float sb)
    {
        const float xa = tb_a * ma, xb = tb_b * mb;
        const float x = xa + xb;
        const float pa = x >= 0.0000001f ? fminf_ordered(xa * __builtin_amdgcn_rcpf(x), 0.999999f) : 0.5f;
        const float pb = 1.f - pa;
        const float nc = fmaf(pa, ba, pb * bb);
        const float va = sa * sa, vb = sb * sb;
        const float da = ba - nc, db = bb - nc;
        const float qa = fmaf(da, da, va), qb = fmaf(db, db, vb);
        const float nv = fmaf(pa, qa, pb * qb);
        const float inv = __builtin_amdgcn_rcpf(nv);
        const float ratio = nv * __builtin_amdgcn_rcpf(sa * sb);
        return fmaf(0.5f, fmaf(qa - nv, inv, (qb - nv) * inv), logf(ratio));
    }

    static __device__ __forceinline__ void merge_values(float tb_a, float tb_b, float ma, float mb, float ba, float bb, float sa, float sb,
        float* nm, float* nc, float* nsd)
    {
        const float xa = tb_a * ma;
        const float xb = tb_b * mb;
        const float pa = (xa + xb >= 0.0000001f) ? fminf_ordered(xa / (xa + xb), 0.999999f) : 0.5f;
        const float pb = 1.f - pa;
        *nc = pa * ba + pb * bb;
        *nm = ma + mb;
        const float va = sa * sa;
        const float vb = sb * sb;
        const float nv = pa * (va + (ba - *nc) * (ba - *nc)) + pb * (vb + (bb - *nc) * (bb - *nc));
        *nsd = sqrt_rn(nv);
    }

    // std::min(a, b) = b < a ? b : a
    static __device__ __forceinline__ float fminf_ordered(float a, float b) { return b < a ? b : a; }

    __device__ __forceinline__ bool full(float threshold) const { return acc >= threshold; }

    // borders of never-filled slots spread evenly up to the furthest relevance end
    __device__ __forceinline__ void finalise()
    {
        float last = 0.f;
#pragma unroll
        for (int i = 0; i < kRasterBins; ++i) {
            const bool inf = __builtin_isinf(b[i]);
            const float kept = larger_of(b[i], last + 0.00001f);
            const float spread = last + (maxd - last) / float(kRasterBins - i);
            b[i] = inf ? spread : kept;
            m[i] = inf ? 0.f : m[i];
            last = b[i];
        }
    }
};

// piecewise_linear::create_approximation for one channel with the left share
// 0.5 (the reference's share is m / (m + m) of one border mass: exactly 0.5,
// and 0/0 -> NaN -> 0.5, vol_raster_forward.cu:450-453)
struct Linear {
    float d0, k0, t1, t2, k2;
};

__device__ __forceinline__ Linear fit_channel(float total, float el, float er, float t_right)
{
    const float m_l = 0.5f * total;
    const float m_r = total - m_l;
    Linear f { el, 0.f, 2.f * m_l / el, t_right - 2.f * m_r / er, 0.f };
    if (total <= 0.000001f)
        return Linear { 0.f, 0.f, 0.f, t_right, 0.f };
    if (f.t2 > f.t1) {
        f.k0 = -el * el / (2.f * m_l);
        f.k2 = er * er / (2.f * m_r);
        return f;
    }
    const float c1 = 2.f * total - (el + er) * t_right;
    const float c2 = er * m_l + el * m_r;
    const float c3 = el * er * t_right;
    const float dm = larger_of(0.f, (c1 + sqrt_rn(c1 * c1 + 4.f * t_right * (2.f * c2 - c3))) / (2.f * t_right));
    float tl, tr;
    if (m_r > m_l) {
        tr = 2.f * m_r / (dm + er);
        tl = larger_of(0.f, t_right - tr);
    } else {
        tl = 2.f * m_l / (dm + el);
        tr = larger_of(0.f, t_right - tl);
    }
    f.k0 = tl == 0.f ? 0.f : -(el - dm) / tl;
    f.t1 = tl;
    f.t2 = tl;
    f.k2 = tr == 0.f ? 0.f : (er - dm) / tr;
    return f;
}

// The channel over the bin's steps, for the integration's inner loop: at step i
// (midpoint (i + 1/2) dt) the value times dt is
//   max(med3(l0 + l1 i, r0 + r1 i, pick), 0)
// of the left and the right segment's lines.  The two segments meet at t1 = t2,
// where the larger line is the one in force if the channel is convex there and
// the smaller if it is concave (pick = +inf, -inf: med3 is their max, min); with
// a gap of zeros between t1 and t2 each line is negative beyond its end, so
// the larger, and 0, is in force.
struct StepLines {
    float l0, l1, r0, r1, pick;
};

__device__ __forceinline__ StepLines step_lines(const Linear& f, float t_right, float dt)
{
    const float base = f.d0 + f.t1 * f.k0; // the right line at t2
    float l0 = f.d0, l1 = f.k0, r0 = base - f.t2 * f.k2, r1 = f.k2;
    const bool apart = f.t2 > f.t1;
    if (apart && f.d0 == 0.f && f.k0 == 0.f && f.k2 == 0.f) {
        r0 = 0.f; // an empty channel
    } else if (apart) {
        r0 = -(f.t2 * f.k2); // the left line ends at 0
    } else if (!(f.t1 > 0.f)) {
        l0 = r0; // no left segment
        l1 = r1;
    } else if (f.k2 == 0.f && !(f.t1 < t_right)) {
        r0 = l0; // no right segment
        r1 = l1;
    }
    const float pick = !apart && f.k0 > f.k2 ? -__builtin_inff() : __builtin_inff();
    const float h = 0.5f * dt;
    return { fmaf(l1, h, l0) * dt, l1 * dt * dt, fmaf(r1, h, r0) * dt, r1 * dt * dt, pick };
}

__device__ __forceinline__ float step_value(const StepLines& c, float i)
{
    return fmaxf(__builtin_amdgcn_fmed3f(fmaf(c.l1, i, c.l0), fmaf(c.r1, i, c.r0), c.pick), 0.f);
}

// The distance from the centre beyond which every bin holds less than the
// 1e-4 that counts (see far_radius in the marcher): z^2 = 2 ln(w 5 750) leaves
// at most 0.87e-4, the rest covers the cdf's rounding (1.2e-7 of w) up to w = 100
__device__ __forceinline__ float raster_far(float w, float var)
{
    const float z2 = 1.3862943611f * (__builtin_amdgcn_logf(w) + 12.4893f);
    const float r = __builtin_amdgcn_sqrtf(fmaxf(z2, 0.f) * var) * 1.0001f;
    return w > 100.f ? __builtin_inff() : r;
}

struct RasterArgs {
    const float* means;
    const float* inv_cov;
    const float* mass;
    const float* rgb;
    const uint32_t* point_list;
    const uint32_t* ranges;
    float inv_proj[16];
    float pos[3];
    float bg[3];
    int width, height, grid_x, grid_y;
    int mode, debug_bin;
    float max_depth;
    float mass_threshold; // -log(transmission_threshold)
    const uint32_t* n_pairs; // device pair count: none leaves the framebuffer untouched
    float* framebuffer;
};

// What a wave knows of the first 64 kSeenWords entries of its tile's list: the
// entries it has tested and those whose mass on every pixel's ray is at most the
// 1e-3 that the rasterisation asks for, which no chunk needs to visit again
constexpr int kSeenWords = 64;

// Where along the tile's rays a Gaussian matters to the bins (gaussian_extent,
// E + z^2 <= 2 ln M + 2 ln 5 750 for raster_far's cut), and how far its density
// at a border is not zero in float (z = 13.5: the last border takes it from
// every Gaussian).  One entry per lane.
struct RasterWindow {
    float lo, hi, trail;
};

__device__ __forceinline__ RasterWindow raster_window(const float* A, float det, const float* m, float mass_norm3, const TileAxis& ax)
{
    const float inf = __builtin_inff();
    const GaussianExtent e = gaussian_extent(A, det, m, mass_norm3, ax);
    if (!e.bounded || !(e.mass < 99.f))
        return RasterWindow { -inf, inf, inf };
    if (e.mass < 0.00099f)
        return RasterWindow { inf, -inf, -inf }; // at most 1e-3 on every ray
    const float half = extent_half(e, 18.f);
    return RasterWindow { e.len - half, e.len + half, e.len + extent_half(e, 185.f) };
}

// Bound by VALU issue.  With every Gaussian's merge costs recomputed over all 32
// slots, every list entry visited for every chunk of 8 bins and the integrand
// evaluated per step, a frame of 200k Gaussians at 1024^2 took 33.4 ms and one of
// 5k at 211x157 8.0 ms; with the merge costs as one logarithm, the windows, bins
// in groups and the integrand's lines 9.9 and 3.1 ms.  16 bins per chunk are what
// two waves per SIMD have registers for.
__global__ __launch_bounds__(kThreads, 2) void k_raster_render(RasterArgs a)
{
    __shared__ float s_mu[3][kThreads];
    __shared__ float s_inv[6][kThreads];
    __shared__ float s_off[3][kThreads]; // mu - camera
    __shared__ float s_norm3[kThreads];
    __shared__ float s_mass[kThreads];
    __shared__ RasterWindow s_win[kThreads];
    __shared__ float s_axis[4];
    __shared__ uint64_t s_seen[kThreads / 64][2][kSeenWords];
    __shared__ float s_rgb[3][kThreads];  // 0 where it is not finite
    __shared__ uint32_t s_odd[kThreads];  // bit c: component c of the colour is infinite (or NaN)
    __shared__ float s_border[kThreads * kBorderStride];
    // the reference returns before rendering when no Gaussian is binned
    // (vol_raster_forward.cu:153-155): the caller's framebuffer stays as it was
    if (*a.n_pairs == 0)
        return;
    const int tile = int(blockIdx.x);
    const int tx = tile % a.grid_x, ty = tile / a.grid_x;
    const int t_id = int(threadIdx.x);
    const int px = tx * kTile + (t_id % kTile), py = ty * kTile + (t_id / kTile);
    const bool inside = px < a.width && py < a.height;
    // ray through the integer pixel coordinate on the near plane (vol_raster_forward.cu:272-278)
    float dir[3];
    {
        const float ndc[3] = { float(px * 2) / float(a.width) - 1.f, float(py * 2) / float(a.height) - 1.f, -1.f };
        float v[4];
        transform_point(a.inv_proj, ndc, v, 4);
        float pv[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            pv[i] = v[i] / v[3] - a.pos[i];
        const float inv_len = 1.f / sqrt_rn(dot3(pv, pv));
#pragma unroll
        for (int i = 0; i < 3; ++i)
            dir[i] = pv[i] * inv_len;
    }
    const TileAxis axis = tile_axis<float>(dir, inside, s_axis);
    const uint32_t first = a.ranges[2 * tile], last = a.ranges[2 * tile + 1];
    const int n_rounds = int((last - first + kThreads - 1) / kThreads);

    int staged = -1; // the batch in LDS (the lists of most tiles fit one)
    const auto stage = [&](int round) {
        if (staged == round)
            return;
        __syncthreads(); // the previous batch has been read
        const uint32_t k = first + uint32_t(round) * kThreads + uint32_t(t_id);
        if (k < last) {
            const uint32_t id = a.point_list[k];
            uint32_t odd = 0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                s_mu[c][t_id] = a.means[3 * id + c];
                const float v = a.rgb[3 * id + c];
                const bool finite = fabsf(v) < __builtin_inff();
                s_rgb[c][t_id] = finite ? v : 0.f;
                odd |= finite ? 0u : 1u << c;
            }
            s_odd[t_id] = odd;
            float A[6];
#pragma unroll
            for (int c = 0; c < 6; ++c)
                s_inv[c][t_id] = A[c] = a.inv_cov[6 * id + c];
            float m[3];
#pragma unroll
            for (int c = 0; c < 3; ++c)
                s_off[c][t_id] = m[c] = s_mu[c][t_id] - a.pos[c];
            const float det = sym3_det(A), norm3 = ray_norm3(det), mass = a.mass[id];
            s_norm3[t_id] = norm3;
            s_mass[t_id] = mass;
            s_win[t_id] = raster_window(A, det, m, mass * norm3, axis);
        }
        __syncthreads();
        staged = round;
    };
    const auto ray1d = [&](int j) {
        const float mu[3] = { s_mu[0][j], s_mu[1][j], s_mu[2][j] };
        const float A[6] = { s_inv[0][j], s_inv[1][j], s_inv[2][j], s_inv[3][j], s_inv[4][j], s_inv[5][j] };
        const float m[3] = { s_off[0][j], s_off[1][j], s_off[2][j] };
        return intersect_ray_pre(mu, A, m, s_norm3[j], a.pos, dir);
    };

    // ---------------------------------------------------------------- pass 1
    BinSizer z;
    z.init();
    if (a.mode != 1) { // Bins mode renders the background only
        bool done = !inside;
        // A pixel's accepted Gaussians wait here, so that one addition to the
        // bins serves pixels that took different Gaussians.  Each is added
        // exactly as if it had been at once; what waits when the bins are full
        // is dropped.
        constexpr int Q = 4;
        float q_mor[Q] = { 0.f, 0.f, 0.f, 0.f }, q_centre[Q] = { 0.f, 0.f, 0.f, 0.f }, q_sd[Q] = { 0.f, 0.f, 0.f, 0.f };
        int waiting = 0;
        for (int r = 0; r < n_rounds; ++r) {
            if (__syncthreads_and(done))
                break;
            stage(r);
            const int count = int(min(uint32_t(kThreads), last - first - uint32_t(r) * kThreads));
            int j = 0;
            while (true) {
                const bool visit = j < count && __builtin_amdgcn_ballot_w64(!done) != 0;
                if (visit) {
                    const Ray1d<float> g = ray1d(j);
                    const float mor = g.weight * s_mass[j];
                    const bool take = !done && !(mor < 0.001f || mor > 1000.f) && !(g.var <= 0.f);
                    const float sd = sqrt_rn(g.var);
                    static_for<Q>([&](auto k) {
                        const bool here = take && waiting == k;
                        q_mor[k] = here ? mor : q_mor[k];
                        q_centre[k] = here ? g.centre : q_centre[k];
                        q_sd[k] = here ? sd : q_sd[k];
                    });
                    waiting += take ? 1 : 0;
                    ++j;
                }
                const int limit = visit ? Q : 1;
                while (__builtin_amdgcn_ballot_w64(waiting >= limit) != 0) {
                    if (waiting > 0) {
                        z.add(q_mor[0], q_centre[0], q_sd[0]);
                        if (z.full(a.mass_threshold)) {
                            done = true;
                            waiting = 1;
                        }
                        --waiting;
                    }
                    static_for<Q - 1>([&](auto k) {
                        q_mor[k] = q_mor[k + 1];
                        q_centre[k] = q_centre[k + 1];
                        q_sd[k] = q_sd[k + 1];
                    });
                }
                if (!visit)
                    break;
            }
        }
        __syncthreads();
        z.finalise();
    }
    // end_of(i): border i, the last one being the furthest relevance end
    float* border = s_border + t_id * kBorderStride;
#pragma unroll
    for (int i = 0; i < kRasterBins - 1; ++i)
        border[i] = z.b[i];
    border[kRasterBins - 1] = z.maxd;
    const auto end_of = [&](int i) { return border[i]; };
    const auto begin_of = [&](int i) { return i == 0 ? 0.f : border[i - 1]; };

    float C[3] = { 0.f, 0.f, 0.f };
    float T = 1.f; // Full mode keeps T = 1: the background is added in full (vol_raster_forward.cu:509-513)
    if (a.mode == 0) {
        // ------------------------------------------------------------ pass 2
        float result[3] = { 0.f, 0.f, 0.f };
        float transparency = 1.f;
        uint32_t odd_seen = 0; // components in which the pixel kept mass of a colour that is not finite
        const float max_distance = end_of(kRasterBins - 1);
        const unsigned lane = lane_id();
        uint64_t* rejected = s_seen[t_id / 64][0];
        uint64_t* known = s_seen[t_id / 64][1];
        rejected[lane] = known[lane] = 0;
        __builtin_amdgcn_wave_barrier();
        for (int k0 = 0; k0 < kRasterBins; k0 += kChunk) {
            float bm[kChunk][4], be[kChunk + 1][4];
            static_for<kChunk>([&](auto q) { bm[q][0] = bm[q][1] = bm[q][2] = bm[q][3] = 0.f; });
            static_for<kChunk + 1>([&](auto q) { be[q][0] = be[q][1] = be[q][2] = be[q][3] = 0.f; });
            const bool last_chunk = k0 + kChunk == kRasterBins;
            // the chunk's borders and, for the bin after it, one more
            const float x_first = begin_of(k0), x_right = end_of(k0 + kChunk - 1);
            const float x_end = last_chunk ? x_right : end_of(k0 + kChunk);
            // the wave's part of the rays
            const float w_first = wave_min(inside ? x_first : __builtin_inff()), w_end = wave_max(inside ? x_end : -__builtin_inff());
            const float w_right = wave_min(inside ? x_right : __builtin_inff());
            for (int r = 0; r < n_rounds; ++r) {
                stage(r);
                const int count = int(min(uint32_t(kThreads), last - first - uint32_t(r) * kThreads));
                for (int j0 = 0; j0 < count; j0 += 64) {
                    const int w_at = (r * kThreads + j0) / 64;
                    const bool tracked = w_at < kSeenWords;
                    uint64_t w_rej = tracked ? uniform_u64(rejected[w_at]) : 0, w_known = tracked ? uniform_u64(known[w_at]) : 0;
                    const RasterWindow win = s_win[min(j0 + int(lane), count - 1)];
                    // beyond the chunk nothing of it counts; before the last
                    // chunk only its density at the last border does
                    const bool met = !(win.lo > w_end) && (!(win.hi < w_first) || (last_chunk && !(win.trail < w_right)));
                    const uint64_t meets = __builtin_amdgcn_ballot_w64(met) & valid_entries(j0, count);
                    for (uint64_t word = meets & ~w_rej; word != 0; word &= word - 1) {
                        const int jj = __builtin_ctzll(word), j = j0 + jj;
                        const Ray1d<float> g = ray1d(j);
                        const float c = g.centre;
                        const float var = g.var;
                        const float w = g.weight * s_mass[j];
                        if (((w_known >> jj) & 1) == 0) {
                            w_known |= uint64_t(1) << jj;
                            if (__builtin_amdgcn_ballot_w64(inside && w > 0.001f) == 0)
                                w_rej |= uint64_t(1) << jj; // the mass within the borders is no larger
                        }
                        const float inv_sd = 1.f / sqrt_rn(var);
                        const float far = raster_far(w, var);
                        bool need = inside && !(var <= 0.f || __builtin_isnan(var) || __builtin_isnan(w) || w > 100000.f);
                        // the last chunk's right border is evaluated for every Gaussian
                        need = need && w > 0.001f && (last_chunk || (c + far > x_first && c - far < x_end));
                        if (__builtin_amdgcn_ballot_w64(need) == 0)
                            continue;
                        // with both ends over 3.1 sd away 0.998 of the mass lies within
                        const bool sure = w > 0.00101f && (max_distance - c) * inv_sd > 3.1f && c * inv_sd > 3.1f;
                        if (__builtin_amdgcn_ballot_w64(need && !sure) != 0)
                            need = need && (sure || !(w * (cdf_sd(c, inv_sd, max_distance) - cdf_sd(c, inv_sd, 0.f)) <= 0.001f));
                        const float lo = need ? c - far : __builtin_inff(), hi = need ? c + far : -__builtin_inff();
                        const float wk = need ? w : 0.f;
                        const float rgb[3] = { s_rgb[0][j], s_rgb[1][j], s_rgb[2][j] };
                        const DensityScale e_scale = density_scale(var);
                        float cdf_start = 0.f;
                        bool have = false, kept = false;
                        static_for<kChunk / kGroup>([&](auto group) {
                            constexpr int g0 = group * kGroup;
                            const float x0 = begin_of(k0 + g0);
                            if (__builtin_amdgcn_ballot_w64(hi > x0 && lo < end_of(k0 + g0 + kGroup - 1)) == 0) {
                                have = false;
                                return;
                            }
                            if (!have)
                                cdf_start = cdf_sd(c, inv_sd, x0);
                            have = true;
                            float x = x0;
                            static_for<kGroup>([&](auto i) {
                                constexpr int q = g0 + i;
                                const float xe = end_of(k0 + q);
                                const float cdf_end = cdf_sd(c, inv_sd, xe);
                                const float mass = (cdf_end - cdf_start) * wk;
                                cdf_start = cdf_end;
                                const bool on = !(mass < 0.0001f) && need;
                                kept = kept || on;
                                const float mq = on ? mass : 0.f;
                                const float d = x - c;
                                const float e = on ? wk * border_density(e_scale, d) : 0.f;
                                x = xe;
                                bm[q][0] = fmaf(rgb[0], mq, bm[q][0]);
                                bm[q][1] = fmaf(rgb[1], mq, bm[q][1]);
                                bm[q][2] = fmaf(rgb[2], mq, bm[q][2]);
                                bm[q][3] += mq;
                                be[q][0] = fmaf(rgb[0], e, be[q][0]);
                                be[q][1] = fmaf(rgb[1], e, be[q][1]);
                                be[q][2] = fmaf(rgb[2], e, be[q][2]);
                                be[q][3] += e;
                            });
                        });
                        // 0 times such a colour is NaN, so it is kept out of the sums
                        const uint32_t odd = __builtin_amdgcn_readfirstlane(s_odd[j]);
                        if (odd != 0)
                            odd_seen |= kept ? odd : 0u;
                        // the evaluation at the chunk's right border belongs to the
                        // next bin, added when that bin's mass passes (or, after the
                        // last bin, always)
                        const bool next = last_chunk ? need : (hi > x_right && lo < x_end);
                        if (__builtin_amdgcn_ballot_w64(next) != 0) {
                            bool add_right = next;
                            if (!last_chunk)
                                add_right = next && !((cdf_sd(c, inv_sd, x_end) - cdf_sd(c, inv_sd, x_right)) * wk < 0.0001f);
                            const float d = x_right - c;
                            const float e = add_right ? wk * border_density(e_scale, d) : 0.f;
                            be[kChunk][0] = fmaf(rgb[0], e, be[kChunk][0]);
                            be[kChunk][1] = fmaf(rgb[1], e, be[kChunk][1]);
                            be[kChunk][2] = fmaf(rgb[2], e, be[kChunk][2]);
                            be[kChunk][3] += e;
                        }
                    }
                    if (tracked && lane == 0) {
                        rejected[w_at] = w_rej;
                        known[w_at] = w_known;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // integrate the chunk's bins (piecewise_linear.h:152-178): per step
            // the channels times dt, the colours weighed with the transparency
            // before the step.  A bin empty on the whole wave changes nothing.
            static_for<kChunk>([&](auto q) {
                const float t_right = end_of(k0 + q) - begin_of(k0 + q);
                const bool some = t_right > 0.f && (bm[q][0] > 0.000001f || bm[q][1] > 0.000001f || bm[q][2] > 0.000001f || bm[q][3] > 0.000001f);
                if (__builtin_amdgcn_ballot_w64(some) == 0)
                    return;
                const float dt = t_right / float(kRasterSteps);
                StepLines f[4];
                static_for<4>([&](auto ch) {
                    f[ch] = some ? step_lines(fit_channel(bm[q][ch], be[q][ch], be[q + 1][ch], t_right), t_right, dt)
                                 : StepLines { 0.f, 0.f, 0.f, 0.f, 0.f };
                });
                float i = 0.f;
#pragma unroll 4
                for (int st = 0; st < kRasterSteps; ++st) {
                    const float e0 = step_value(f[0], i), e1 = step_value(f[1], i), e2 = step_value(f[2], i), e3 = step_value(f[3], i);
                    result[0] = fmaf(e0, transparency, result[0]);
                    result[1] = fmaf(e1, transparency, result[1]);
                    result[2] = fmaf(e2, transparency, result[2]);
                    transparency *= fmaxf(1.f - e3, 0.f);
                    i += 1.f;
                }
            });
        }
#pragma unroll
        for (int ch = 0; ch < 3; ++ch)
            C[ch] = (odd_seen >> ch) & 1u ? __builtin_nanf("") : result[ch];
    } else if (a.mode == 2) {
        const int bin = int(min(unsigned(a.debug_bin), unsigned(kRasterBins - 1)));
        const float dist = end_of(bin);
        const float v = dist / a.max_depth;
        C[0] = C[1] = C[2] = v;
        if (dist == 0.f) {
            C[0] = 0.f;
            C[1] = 1.f;
            C[2] = 0.f;
        }
        if (__builtin_isnan(dist)) {
            C[0] = 1.f;
            C[1] = 0.f;
            C[2] = 0.5f;
        }
        if (dist < 0.f) {
            C[0] = 1.f;
            C[1] = 0.5f;
            C[2] = 0.f;
        }
        T = 0.f;
    }
    if (!inside)
        return;
    const int64_t plane = int64_t(a.width) * a.height;
    const int64_t q = int64_t(py) * a.width + px;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
        a.framebuffer[ch * plane + q] = C[ch] + T * a.bg[ch];
}

} // namespace
} // namespace dgmr

using namespace dgmr;

extern "C" {

int dgmr_raster_forward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_raster_options* opt, dgmr_splat_geometry* geom,
    dgmr_binning* bins, float* inv_cov, float* mass, float* framebuffer, void* workspace, size_t workspace_bytes, dgmr_stats* stats,
    dgmr_stream stream)
{
    DGMR_ARG_CHECK(g && cam && opt && geom && bins && inv_cov && mass && framebuffer && workspace, "dgmr_raster_forward: null argument");
    DGMR_ARG_CHECK(g->dtype == DGMR_F32, "dgmr_raster_forward: the rasteriser computes in float32");
    DGMR_ARG_CHECK(g->n >= 0 && g->n < (int64_t(1) << 31), "dgmr_raster_forward: bad Gaussian count");
    DGMR_ARG_CHECK(g->sh_coeffs >= 1 && g->sh_coeffs <= 16 && g->sh_degree >= 0 && g->sh_degree <= 3, "dgmr_raster_forward: bad SH layout");
    DGMR_ARG_CHECK(valid_image(cam->width, cam->height), "dgmr_raster_forward: bad image size");
    DGMR_ARG_CHECK(opt->render_mode >= 0 && opt->render_mode <= 2, "dgmr_raster_forward: render mode must be 0 (full), 1 (bins) or 2 (depth)");
    DGMR_ARG_CHECK(bins->point_list && bins->ranges, "dgmr_raster_forward: null binning buffers");
    const int64_t n = g->n;
    DGMR_ARG_CHECK(workspace_bytes >= splat_workspace_bytes(n, bins->pair_capacity), "dgmr_raster_forward: workspace too small");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const dgmr_tiling tiling { kTile, kTile, 64, 0, 0 }; // the reference's rectangles
    const DevCamera<float> dc = make_dev_camera<float>(*cam, tiling);
    const int64_t n_tiles = int64_t(dc.grid_x) * dc.grid_y;
    if (stats) {
        stats->n_pairs = 0;
        stats->n_visible = 0;
    }
    RasterArgs ra {};
    ra.means = static_cast<const float*>(g->means);
    ra.inv_cov = inv_cov;
    ra.mass = mass;
    ra.rgb = geom->rgb;
    ra.point_list = bins->point_list;
    ra.ranges = bins->ranges;
    for (int i = 0; i < 16; ++i)
        ra.inv_proj[i] = dc.inv_proj[i];
    for (int i = 0; i < 3; ++i) {
        ra.pos[i] = dc.pos[i];
        ra.bg[i] = dc.bg[i];
    }
    ra.width = cam->width;
    ra.height = cam->height;
    ra.grid_x = dc.grid_x;
    ra.grid_y = dc.grid_y;
    ra.mode = opt->render_mode;
    ra.debug_bin = opt->debug_bin;
    ra.max_depth = opt->max_depth;
    ra.mass_threshold = float(-std::log(double(0.005f))); // -log(vol_raster::config::transmission_threshold)
    ra.framebuffer = framebuffer;
    if (n == 0) {
        // nothing binned: the reference returns before rendering, the framebuffer is left as it was
        DGMR_HIP_CHECK(hipMemsetAsync(bins->ranges, 0, size_t(n_tiles) * 2 * sizeof(uint32_t), st));
        return DGMR_OK;
    }
    uint32_t *dkeys, *dids;
    uint2* brects;
    binning_key_buffers(workspace, n, false, &dkeys, &dids, reinterpret_cast<void**>(&brects));
    {
        StageScope sc("raster.preprocess", st, double(n) * (44.0 + 12.0 * g->sh_coeffs + 75.0 + 28.0));
        DGMR_HIP_CHECK(launch_splat_preprocess(g, dc,
            SplatOut { geom->rects, geom->tiles_touched, geom->xy, reinterpret_cast<float4*>(geom->conic_opacity), geom->rgb, geom->rgb_clamped,
                geom->depths, dkeys, dids, brects, nullptr },
            st));
        k_raster_extra<<<unsigned(ceil_div64(n, 256)), 256, 0, st>>>(n, make_splat_params(g), dc, geom->tiles_touched, inv_cov, mass);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    Carver cv(workspace, workspace_bytes);
    PendingCount pending;
    const int rc = bin_gaussians(n, geom->rects, geom->tiles_touched, geom->xy, false, true, false, dc.grid_x, dc.grid_y, dc.tile_w, dc.tile_h, bins, cv,
        &pending, st, nullptr);
    if (rc != DGMR_OK)
        return rc;
    ra.n_pairs = pending.device;
    {
        StageScope sc("raster.render", st);
        k_raster_render<<<unsigned(n_tiles), kThreads, 0, st>>>(ra);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    const int64_t R = pending.wait();
    if (R < 0)
        return DGMR_ERR_DEVICE;
    if (stats)
        stats->n_pairs = R;
    if (R > bins->pair_capacity) {
        set_error("pair capacity too small");
        return DGMR_ERR_CAPACITY;
    }
    return DGMR_OK;
}

} // extern "C"
