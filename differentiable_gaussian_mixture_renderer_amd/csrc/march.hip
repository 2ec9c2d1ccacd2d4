// SPDX-License-Identifier: GPL-3.0-or-later
// Volumetric ray marcher for gfx950, float and double (reference:
// src/dgmr/vol_marcher_forward.cu:42-503, vol_marcher_backward.cu:53-386).
//
// Per pixel (one thread; a block is one tile), each large step:
//   pass 1  build up to 16 sample sections from the tile's depth-ordered
//           Gaussians (sampling density = 31 steps over +-3 sigma of each)
//   pass 2  deposit every Gaussian's ray mass into 127 bins between 128
//           borders placed by the sections (erf-based, per bin)
//   blend   C += rgb_m T, T *= exp(-m) per bin
// The reference keeps 128 borders and 127 vec4 bins per thread (2.7 KB in
// float), beyond the 512-VGPR budget of a CDNA4 lane.  Here the bins are
// processed in register-sized chunks: borders are generated by a walk over the
// sections, each chunk's bins are filled by a pass over the tile's Gaussians
// and blended before the next chunk, carrying (C, T).  Per-bin accumulation
// order over Gaussians is unchanged, so each bin holds the same value.  The
// backward replays the march, recomputing transmittance, and pushes each
// chunk's adjoint through the ray restriction (linear in the 1D adjoints),
// summing over the 64 pixels of a wave before the atomics.  Given a replay
// store (device memory of about 2.5 KB per pixel and large step), the forward
// also writes every chunk's bins and borders, and the backward reads them
// back instead of recomputing sections and bins: only the adjoint walks
// remain (200k Gaussians at 1024^2, all steps kept: 11.2 ms against 26.0
// recomputed and 16.7 forward).
#include <algorithm>
#include <utility>

#include "host_common.h"
#include "march_device.h"
#include "primitives.h"

namespace dgmr {

namespace {

constexpr int kPreThreads = 256;

template <class S>
struct MarchArgs {
    const S* means;
    const S* scales;
    const S* rotations;
    const S* opacity;
    const S* sh;
    int sh_coeffs, sh_degree;
    S scale_multiplier;
};

// vol_marcher_forward.cu:98-176.  Binning decisions (culling, mass <= 0,
// iso-line rect, tiles, depth key) use the same operation sequence as the host
// restatement.
template <class S>
__global__ __launch_bounds__(kPreThreads) void k_march_preprocess(int64_t n, MarchArgs<S> a, DevCamera<S> cam, int32_t* __restrict__ rects,
    uint32_t* __restrict__ tiles, S* __restrict__ xy_out, S* __restrict__ depths, S* __restrict__ rgb_out, uint8_t* __restrict__ clamped_out,
    S* __restrict__ inv_cov_out, S* __restrict__ mass_out, uint32_t* __restrict__ depth_keys, uint32_t* __restrict__ ids)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    tiles[i] = 0;
    rects[2 * i] = 0;
    rects[2 * i + 1] = 0;
    xy_out[2 * i] = 0;
    xy_out[2 * i + 1] = 0;
    depth_keys[i] = 0xffffffffu;
    if (ids) // null when the binning's compaction numbers the entries
        ids[i] = uint32_t(i);
    const S mu[3] = { a.means[3 * i], a.means[3 * i + 1], a.means[3 * i + 2] };
    S t[3];
    transform_point(cam.view, mu, t, 3);
    if (t[2] < S(0.2f))
        return;
    const S w = a.opacity[i];
    const S m = a.scale_multiplier;
    const S s[3] = { a.scales[3 * i] * m, a.scales[3 * i + 1] * m, a.scales[3 * i + 2] * m };
    const S q[4] = { a.rotations[4 * i], a.rotations[4 * i + 1], a.rotations[4 * i + 2], a.rotations[4 * i + 3] };
    const S dv[3] = { cam.pos[0] - mu[0], cam.pos[1] - mu[1], cam.pos[2] - mu[2] };
    const S dist = length3(dv);
    S cov[6];
    compute_cov(s, q, cov);
    const S aa = div_rn(S(kFilterSD) * cam.tan_fovx * S(2), S(cam.width));
    const S f = dist * aa;
    const S f2 = f * f;
    const S cov_f[6] = { cov[0] + f2, cov[1], cov[2], cov[3] + f2, cov[4], cov[5] + f2 };
    S W[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            W[r][c] = cam.view[4 * c + r];
    S c2[3];
    affine_cut(cov, W, c2);
    const S mass = w * (S(2 * kPi) * sqrt_rn(c2[0] * c2[2] - c2[1] * c2[1]));
    if (mass <= 0)
        return;
    // splat<Opacity> with a 0.55^2 px filter for the iso-line rect
    SplatIn<S> in;
    splat_internals(mu, s, q, cam, &in);
    const S filt = S(kFilterSD * kFilterSD);
    const S sc[3] = { in.cov2[0] + filt, in.cov2[1], in.cov2[2] + filt };
    const S det_c = in.cov2[0] * in.cov2[2] - in.cov2[1] * in.cov2[1];
    const S det_n = sc[0] * sc[2] - sc[1] * sc[1];
    const S wt = w * sqrt_rn(dmax(S(0.000025), div_rn(det_c, det_n)));
    S xy[2];
    project_to_screen(mu, cam, xy);
    const S level = S(1.f / 255.f);
    const S iso_v = S(-2) * portable_log(div_rn(level, wt));
    const S ex = iso_v <= 0 ? S(0) : sqrt_rn(iso_v * sc[0]);
    const S ey = iso_v <= 0 ? S(0) : sqrt_rn(iso_v * sc[2]);
    const int ext_x = guarded_int(dceil(ex));
    const int ext_y = guarded_int(dceil(ey));
    rects[2 * i] = ext_x;
    rects[2 * i + 1] = ext_y;
    int x0, y0, x1, y1;
    get_rect(xy[0], xy[1], ext_x, ext_y, cam.grid_x, cam.grid_y, cam.tile_w, cam.tile_h, &x0, &y0, &x1, &y1);
    const uint32_t touched = uint32_t(x1 - x0) * uint32_t(y1 - y0);
    if (touched == 0)
        return;
    tiles[i] = touched;
    xy_out[2 * i] = xy[0];
    xy_out[2 * i + 1] = xy[1];
    S inv[6];
    sym3_inverse(cov_f, inv);
#pragma unroll
    for (int k = 0; k < 6; ++k)
        inv_cov_out[6 * i + k] = inv[k];
    const S depth = dist - div_rn(dmax(s[0], dmax(s[1], s[2])) * S(kRelevanceSigma), S(2));
    depths[i] = depth;
    depth_keys[i] = __float_as_uint(float(depth));
    const S dir[3] = { div_rn(-dv[0], dist), div_rn(-dv[1], dist), div_rn(-dv[2], dist) };
    S Y[16];
    sh_basis(a.sh_degree, dir, Y);
    const int kmax = min(a.sh_coeffs, (a.sh_degree + 1) * (a.sh_degree + 1));
    const S* c = a.sh + i * a.sh_coeffs * 3;
    // all coefficient loads in flight before the first product (one at a
    // time, each would wait for its load)
    S cf[48];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const bool on = k < kmax;
        cf[3 * k + 0] = on ? c[3 * k + 0] : S(0);
        cf[3 * k + 1] = on ? c[3 * k + 1] : S(0);
        cf[3 * k + 2] = on ? c[3 * k + 2] : S(0);
    }
    S r0 = 0, r1 = 0, r2 = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k < kmax) {
            r0 += Y[k] * cf[3 * k + 0];
            r1 += Y[k] * cf[3 * k + 1];
            r2 += Y[k] * cf[3 * k + 2];
        }
    }
    r0 += S(0.5);
    r1 += S(0.5);
    r2 += S(0.5);
    rgb_out[3 * i + 0] = dmax(r0, S(0));
    rgb_out[3 * i + 1] = dmax(r1, S(0));
    rgb_out[3 * i + 2] = dmax(r2, S(0));
    clamped_out[3 * i + 0] = r0 >= S(0);
    clamped_out[3 * i + 1] = r1 >= S(0);
    clamped_out[3 * i + 2] = r2 >= S(0);
    mass_out[i] = mass;
}

// A Gaussian of the tile's list in LDS: what the passes read at one address for
// the whole wave, with the per-Gaussian parts of the ray restriction (centre
// relative to the camera, normalisation) computed once when it is staged
// instead of by every pixel of every pass.
template <class S>
struct alignas(16) Staged {
    S A[6];   // inverse filtered covariance
    S m[3];   // mu - o
    S mu[3];
    S norm3;  // sqrt(det A) / sqrt((2 pi)^3)
    S mass;
    S rgb[3];     // 0 where it is not finite
    S depth;
    uint32_t id;
    uint32_t odd; // bit c: component c of the colour is infinite or NaN, bit 3 + c: NaN
};

template <class S>
__device__ __forceinline__ Ray1d<S> intersect_staged(const Staged<S>& g, const S* o, const S* d)
{
    return intersect_ray_pre(g.mu, g.A, g.m, g.norm3, o, d);
}

// The window of a Gaussian over the tile's rays (gaussian_extent): a section or
// a bin of it needs
//   mass on the ray >= 1/255 and z <= 3:   E + z^2 <= 2 ln M + 2 ln 255 + 9
//   z within far_radius' cut:              E + z^2 <= 2 ln M + 2 ln 55556, or
//                                          + 5.5^2 - 2 ln 2 when M can exceed 2
// and with M >= 10 (never cut) it is the whole axis.
template <class S>
__device__ __forceinline__ Reach1d ray_window(const Staged<S>& g, S detA, const TileAxis& ax)
{
    const float inf = __builtin_inff();
    const float A[6] = { float(g.A[0]), float(g.A[1]), float(g.A[2]), float(g.A[3]), float(g.A[4]), float(g.A[5]) };
    const float m[3] = { float(g.m[0]), float(g.m[1]), float(g.m[2]) };
    const GaussianExtent e = gaussian_extent(A, float(detA), m, float(g.mass) * float(g.norm3), ax);
    if (!e.bounded || !(e.mass < 9.9f))
        return Reach1d { -inf, inf };
    if (e.mass < 0.0039f)
        return Reach1d { inf, -inf }; // under 1/255 on every ray
    const float half = extent_half(e, e.mass > 1.9f ? 29.f : 22.f);
    return Reach1d { e.len - half, e.len + half };
}

template <class S>
struct MarchData;

template <class S>
__device__ __forceinline__ void stage_gaussian(Staged<S>* dst, Reach1d* win, uint32_t id, const MarchData<S>& md, const S* o, const TileAxis& ax);

struct MarchControl {
    int max_large_steps;
    int n_frozen;
    double frozen[8][3];
    int bins_per_chunk; // bins held in registers per pass over a tile's Gaussians (float: 16 or 32)
    int render_mode;    // 0 full, 1 bins, 2 depth (forward only)
    int debug_bin;
    double max_depth;
};

template <class S>
struct MarchData {
    const uint32_t* ranges;
    const uint32_t* point_list;
    const S* means;
    const S* inv_cov;
    const S* rgb;
    const S* mass;
    const S* depths;
    int n_tiles;
    const uint32_t* n_pairs; // device pair count (forward); null: pairs exist
};

// Replay store: what the forward integrated, kept for the backward.  Per tile
// and kept large step one record of replay_record_elems<NT>() elements: the
// 127 bins of every pixel ([bin][pixel][rgb mass, mass]), the 128 bin borders
// ([border][pixel]) and whether the pixel marched that step ([pixel], 1 or
// 0); per tile the number of large steps its block took (kReplayNotKept when
// the forward kept nothing for it).
template <class S>
struct Replay {
    S* data;
    uint32_t* tile_steps;
    int steps; // large steps kept per tile; 0: no store
};

constexpr uint32_t kReplayNotKept = 0xffffffffu;

template <class S>
__device__ __forceinline__ void stage_gaussian(Staged<S>* dst, Reach1d* win, uint32_t id, const MarchData<S>& md, const S* o, const TileAxis& ax)
{
    Staged<S> g;
    g.odd = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g.mu[k] = md.means[3 * id + k];
        const S c = md.rgb[3 * id + k];
        const bool odd = !(fabs(c) < S(__builtin_huge_val()));
        g.rgb[k] = odd ? S(0) : c;
        g.odd |= odd ? (c != c ? 9u : 1u) << k : 0u;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k)
        g.A[k] = md.inv_cov[6 * id + k];
    g.mass = md.mass[id];
    g.depth = md.depths[id];
    g.id = id;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        g.m[k] = g.mu[k] - o[k];
    const S detA = sym3_det(g.A);
    g.norm3 = ray_norm3(detA);
    *win = ray_window(g, detA, ax);
    *dst = g;
}

template <int NT>
__host__ __device__ constexpr int64_t replay_record_elems()
{
    return int64_t(NT) * (4 * kBins + kBorders + 1);
}

template <class S>
__device__ __forceinline__ void store4(S* p, S a, S b, S c, S d)
{
    p[0] = a;
    p[1] = b;
    p[2] = c;
    p[3] = d;
}

template <>
__device__ __forceinline__ void store4<float>(float* p, float a, float b, float c, float d)
{
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
}

// A copy the compiler does not trace back: a 16-byte store needs four
// consecutive registers, and without it the bins would be held that way (and
// copied) through the whole deposit loop.
__device__ __forceinline__ float detached(float v)
{
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ double detached(double v) { return v; }

template <class S>
__device__ __forceinline__ void load4(const S* p, S* v)
{
    v[0] = p[0];
    v[1] = p[1];
    v[2] = p[2];
    v[3] = p[3];
}

template <>
__device__ __forceinline__ void load4<float>(const float* p, float* v)
{
    const float4 q = *reinterpret_cast<const float4*>(p);
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    v[3] = q.w;
}

__device__ __forceinline__ int xcd_tile_m(int b, int n_tiles)
{
    const int q = n_tiles / 8, r = n_tiles % 8;
    const int x = b % 8, slot = b / 8;
    return x * q + min(x, r) + slot;
}

// A Gaussian on this pixel's ray: centre, 1 / sd, mass on the ray, and the
// distance from the centre beyond which every bin holds less than 1e-5 (the
// reference's per-bin threshold, so bins out there take nothing).
template <class S>
struct RayGauss {
    S centre, inv_sd, mor, far;
};

// The far distance: the tail beyond z sd holds at most exp(-z^2 / 2) / 2 of the
// mass, so z^2 = 2 ln(mor / 1.8e-5) leaves every bin there at most 0.9e-5; the
// rest of the 1e-5 covers the float cdf's 1.5e-7 (twice, for mor <= 2).  Above
// that 5.5 sd, and no cut for more than 10 (which could reach 1e-5 by the
// cdf's error alone).
__device__ __forceinline__ float far_radius(float mor, float var)
{
    const float z2 = 1.3862943611f * (__builtin_amdgcn_logf(mor) + 15.7616f); // 2 ln2 (log2 mor + log2 55556)
    const float r = __builtin_amdgcn_sqrtf((mor > 1.99f ? 30.25f : z2) * var);
    return mor > 9.99f ? __builtin_inff() : r;
}

// A restricted to the ray and whether it can deposit mass (math.h:436-454)
template <class S>
__device__ __forceinline__ bool ray_gaussian(const Staged<S>& g, const S* o, const S* d, RayGauss<S>* out)
{
    const Ray1d<S> r = intersect_staged(g, o, d);
    const S sd = sqrt_rn(r.var);
    out->centre = r.centre;
    out->inv_sd = S(1) / sd;
    out->mor = r.weight * g.mass;
    out->far = S(far_radius(float(out->mor), float(r.var)) * 1.00001f);
    if (r.centre != r.centre)
        return false;
    if (out->mor < S(1.0f / 255.f) || out->mor > S(1000))
        return false;
    if (sd <= S(0.0001) || sd != sd || out->mor != out->mor)
        return false;
    return true;
}

// Per-wave candidate masks over the tile's list: the Gaussian at list
// position p is a candidate when it passes the mass-on-ray test (1/255 <=
// mass <= 1000, or NaN) on some pixel of the wave.  One that fails it on every
// pixel deposits nothing (math.h:440-443) and has no adjoint, so the passes of
// every large step skip it for the whole wave.  The test does not depend on the
// large step: the first pass that visits an entry evaluates its restriction
// anyway, and records the answer in LDS.  Positions from kCandEntries on are
// not recorded and always taken.
constexpr int kCandWords = 64;
constexpr uint32_t kCandEntries = 64u * kCandWords;

// a wave's words, in LDS: bit p of `rejected` is set once position p is known
// not to be a candidate, bit p of `known` once it was tested
struct Candidates {
    uint64_t* rejected;
    uint64_t* known;
};

// the 64-entry word at a list position, while a pass visits its entries
struct CandidateWord {
    uint64_t rejected, known;
    int at; // -1: not recorded

    __device__ __forceinline__ CandidateWord(const Candidates& c, uint32_t pos) : rejected(0), known(0), at(-1)
    {
        if (pos < kCandEntries) {
            at = int(pos / 64);
            rejected = uniform_u64(c.rejected[at]);
            known = uniform_u64(c.known[at]);
        }
    }
    // entry j was visited; mor: its mass on the lane's ray
    template <class S>
    __device__ __forceinline__ void visited(int j, bool inside, S mor)
    {
        const uint64_t bit = uint64_t(1) << j;
        if ((known & bit) == 0) {
            known |= bit;
            if (__builtin_amdgcn_ballot_w64(inside && !(mor < S(1.0f / 255.f)) && !(mor > S(1000))) == 0)
                rejected |= bit;
        }
    }
    __device__ __forceinline__ void store(const Candidates& c) const
    {
        if (at >= 0 && lane_id() == 0) {
            c.rejected[at] = rejected;
            c.known[at] = known;
        }
        __builtin_amdgcn_wave_barrier(); // LDS operations of a wave execute in order: later reads see the word
    }
};

// clears a wave's words; every lane of the wave calls it
__device__ __forceinline__ Candidates clear_candidates(uint64_t (*words)[kCandWords])
{
    words[0][lane_id()] = 0;
    words[1][lane_id()] = 0;
    __builtin_amdgcn_wave_barrier();
    return { words[0], words[1] };
}
static_assert(kCandWords == 64, "one word per lane");

// The tile's list in LDS, NT entries at a time, for the block's passes over it
template <class S, int NT>
struct TileList {
    Staged<S>* s_g;
    Reach1d* s_win;
    const MarchData<S>& md;
    uint32_t first, last;
    TileAxis axis;
    uint32_t staged; // first entry of the staged batch; last: none

    // stages the batch at `base` unless it is there already (the lists of most
    // tiles fit one batch); every thread of the block calls it
    __device__ __forceinline__ void stage(uint32_t base, const S* o)
    {
        if (staged == base)
            return;
        __syncthreads(); // the previous batch has been read
        const uint32_t k = base + threadIdx.x;
        if (k < last)
            stage_gaussian(&s_g[threadIdx.x], &s_win[threadIdx.x], md.point_list[k], md, o, axis);
        __syncthreads();
        staged = base;
    }
};

// The tile's section lists, in LDS: indexed at run time by the border walk,
// and (in the in-order insertion) by the list itself, they would live in private
// memory as a thread's own array.  52 KB for a 256-pixel tile in float, which
// two workgroups per CU hold beside their staging; 104 KB in double, one
// workgroup per CU, which is what the double kernels' registers allow.
template <class S, int NT>
struct SectionSmem {
    S words[3 * SectionStore<S, kSections, NT>::kSlots * NT];
};

template <class S, int NT>
__device__ __forceinline__ SectionList<S, kSections, NT> section_list(SectionSmem<S, NT>& sm)
{
    SectionList<S, kSections, NT> sec;
    sec.data.base = sm.words + threadIdx.x;
    return sec;
}

// Whether the section pass may visit only the wave's candidates: a Gaussian
// that fails the mass-on-ray test on every pixel of the wave adds no section
// there, and skipping it cannot move the depth break as long as depth never
// decreases along the tile's list (the section list does not change in
// between, so the break falls at the next visited Gaussian instead).  The list
// is ordered by the float32 depth bits: depths ascend up to the first
// negative or NaN one, and those sort last, so the last entry tells.  The
// double path keeps the full walk (its depths are ordered by their float32
// rounding only).
template <class S>
__device__ __forceinline__ bool sections_by_candidates(const MarchData<S>& md, uint32_t first, uint32_t last)
{
    if (sizeof(S) != 4 || first >= last)
        return false;
    const float dl = float(md.depths[md.point_list[last - 1]]);
    return !((__float_as_uint(dl) >> 31) || dl != dl);
}

// pass 1: sample sections from the tile's Gaussians (vol_marcher_forward.cu:350-403).
// by_cand: visit only the candidates whose window meets the part of the ray
// between the step's start and the list's end (a section outside it is not
// put; the depth break moves as for the candidates)
template <class S, int NT, class L>
__device__ __forceinline__ void build_sections(L& sec, TileList<S, NT>& tl, bool skip, bool inside, const S* o, const S* d, const MarchControl& ctl,
    bool by_cand, const Candidates& cand)
{
    if (ctl.n_frozen > 0) {
        for (int k = 0; k < ctl.n_frozen; ++k)
            sec.put({ S(ctl.frozen[k][0]), S(ctl.frozen[k][1]), S(ctl.frozen[k][2]) });
        return;
    }
    bool done1 = skip;
    const float wlo = by_cand ? wave_min(skip ? __builtin_inff() : float(sec.start_)) : 0.f;
    // A pixel's accepted Gaussians wait here, so that one insertion serves
    // pixels that took different Gaussians (a wave visits about 50 Gaussians
    // per large step, a pixel takes a third of them).  Each is inserted, or
    // stops the pass, exactly as if it had been at once: its depth is held
    // against the list's end when its turn comes.
    constexpr int Q = 4;
    S q_centre[Q], q_sd[Q], q_depth[Q];
    int waiting = 0;
    static_for<Q>([&](auto k) { q_centre[k] = q_sd[k] = q_depth[k] = 0; });
    for (uint32_t base = tl.first; base < tl.last; base += NT) {
        if (__syncthreads_count(!done1) == 0)
            break;
        tl.stage(base, o);
        // the batch's first Gaussian is its shallowest: past it, every later
        // one is beyond the list's end too (the break the full walk takes)
        if (sec.end_ < tl.s_g[0].depth)
            done1 = true;
        const int cnt = int(min<uint32_t>(NT, tl.last - base));
        int j0 = -64;
        uint64_t word = 0;
        CandidateWord cw(cand, kCandEntries);
        while (true) {
            while (word == 0 && j0 + 64 < cnt) {
                j0 += 64;
                cw.store(cand);
                cw = CandidateWord(cand, base - tl.first + uint32_t(j0));
                word = valid_entries(j0, cnt);
                if (by_cand)
                    word = entries_in(tl.s_win, j0, cnt, wlo, wave_max(done1 ? -__builtin_inff() : float(sec.end_))) & ~cw.rejected;
            }
            const bool visit = word != 0 && __builtin_amdgcn_ballot_w64(!done1) != 0;
            if (visit) {
                const int j = __builtin_ctzll(word);
                const Staged<S>& g = tl.s_g[j0 + j];
                word &= word - 1;
                if (sec.end_ < g.depth)
                    done1 = true;
                const Ray1d<S> r = intersect_staged(g, o, d);
                const S mor = r.weight * g.mass;
                cw.visited(j, inside, mor);
                const S sd = sqrt_rn(r.var), half = sd * S(kRelevanceSigma);
                const bool out = r.centre + half <= sec.start_ || r.centre - half >= sec.end_; // put would return
                const bool take = !done1 && !(mor <= S(1.0f / 255.f) || mor > S(1000)) && !(r.var <= 0) && r.centre == r.centre && !out;
                static_for<Q>([&](auto k) {
                    const bool here = take && waiting == k;
                    q_centre[k] = here ? r.centre : q_centre[k];
                    q_sd[k] = here ? sd : q_sd[k];
                    q_depth[k] = here ? g.depth : q_depth[k];
                });
                waiting += take ? 1 : 0;
            }
            // a full walk (depths not ascending) inserts at once; so does the
            // end of a batch
            const int limit = visit && by_cand ? Q : 1;
            while (__builtin_amdgcn_ballot_w64(waiting >= limit) != 0) {
                if (waiting > 0) {
                    if (sec.end_ < q_depth[0]) {
                        done1 = true;
                        waiting = 1; // the later ones are deeper
                    } else {
                        const S half = q_sd[0] * S(kRelevanceSigma);
                        sec.put({ q_centre[0] - half, q_centre[0] + half, (q_sd[0] * S(kRelevanceSigma) * S(2)) / S(kStepsPerGaussian - 1) });
                    }
                    --waiting;
                }
                static_for<Q - 1>([&](auto k) {
                    q_centre[k] = q_centre[k + 1];
                    q_sd[k] = q_sd[k + 1];
                    q_depth[k] = q_depth[k + 1];
                });
            }
            if (!visit)
                break;
        }
        cw.store(cand);
    }
}

// A lane's share of one Gaussian in the chunk [bb[0], bb[CB]]: whether it can
// deposit there at all.  The mass within the step's bins must reach 1e-4
// (math.h:455-460): with at least 1/255 on the ray that is certain when the
// centre lies in the bins, 0.1 sd from one of their ends (0.04 of the mass);
// otherwise the cdf at both ends decides.
template <class S>
__device__ __forceinline__ bool deposits_in(const RayGauss<S>& r, bool pass, S b_first, S b_last, S lo, S hi)
{
    bool need = pass && r.centre + r.far > lo && r.centre - r.far < hi;
    const S zl = (b_last - r.centre) * r.inv_sd, zf = (b_first - r.centre) * r.inv_sd;
    const bool sure = (zl > S(0.1) && zf <= S(0)) || (zl >= S(0) && zf < S(-0.1));
    if (__builtin_amdgcn_ballot_w64(need && !sure) != 0) {
        const S in_bins = r.mor * (cdf_inv_sd(r.centre, r.inv_sd, b_last) - cdf_inv_sd(r.centre, r.inv_sd, b_first));
        need = need && (sure || !(in_bins < S(0.0001f)));
    }
    return need;
}

// Bins per group: a wave evaluates the groups of a chunk that some lane's
// Gaussian reaches (far_radius), the others hold less than 1e-5 per bin
constexpr int kBinGroup = 8;

// pass 2 for one chunk of bins [bb[0], bb[CB]] (borders past the chunk's last
// bin repeat its end, so the bins there are empty): every Gaussian of the tile
// deposits its ray mass (math.h:430-468), in tile order; pixels with `stopped`
// take part in the block's staging only.  Only the entries whose window meets
// the wave's part of the chunk are visited, and only the wave's candidates of
// them.  Bound by VALU issue.  Visiting every candidate in every chunk, with
// the exact restriction each time and all of a chunk's bins once one pixel's
// Gaussian reached it, the forward took 52.0 ms on 200k Gaussians at 1024^2 and
// forward + backward 56.3 ms on 60k at 491x373; with windows, groups and the
// sections of sections.h 17.7 and 24.0 ms.
template <bool ODD, class S, int NT, int CB>
__device__ __forceinline__ void fill_chunk(S (&bins)[CB][4], const S (&bb)[CB + 1], bool stopped, TileList<S, NT>& tl, bool inside,
    const S* o, const S* d, S b_first, S b_last, const Candidates& cand)
{
#pragma unroll
    for (int k = 0; k < CB; ++k)
        bins[k][0] = bins[k][1] = bins[k][2] = bins[k][3] = 0;
    // ODD: a colour that is not finite goes only where its mass does (0 times it
    // is NaN): the bins, as bits per component, that kept mass of such a colour.
    // The backward needs none of it: the pixel's own colour is not finite.
    uint32_t odd_bins[3] = { 0, 0, 0 }, odd_nan = 0;
    static_assert(CB <= 32, "one bit per bin");
    const uint32_t end = __syncthreads_count(!stopped) == 0 ? tl.first : tl.last;
    const float inf = __builtin_inff();
    // no entry meets the empty window of a wave whose pixels have all stopped
    const float wlo = wave_min(stopped ? inf : float(bb[0])), whi = wave_max(stopped ? -inf : float(bb[CB]));
    for (uint32_t base = tl.first; base < end; base += NT) {
        tl.stage(base, o);
        const int cnt = int(min<uint32_t>(NT, tl.last - base));
        for (int j0 = 0; j0 < cnt; j0 += 64) {
            uint64_t word = entries_in(tl.s_win, j0, cnt, wlo, whi);
            if (word == 0)
                continue;
            CandidateWord cw(cand, base - tl.first + uint32_t(j0));
            for (word &= ~cw.rejected; word != 0; word &= word - 1) {
                const int j = __builtin_ctzll(word);
                const Staged<S>& g = tl.s_g[j0 + j];
                RayGauss<S> r;
                const bool pass = ray_gaussian(g, o, d, &r) && !stopped;
                cw.visited(j, inside, r.mor);
                if (__builtin_amdgcn_ballot_w64(pass && r.centre + r.far > bb[0] && r.centre - r.far < bb[CB]) == 0)
                    continue;
                const bool need = deposits_in(r, pass, b_first, b_last, bb[0], bb[CB]);
                const S lo = need ? r.centre - r.far : S(inf), hi = need ? r.centre + r.far : S(-inf);
                const S mor = need ? r.mor : S(0);
                if constexpr (ODD) {
                    const uint32_t odd = __builtin_amdgcn_readfirstlane(g.odd);
                    if (odd != 0) {
                        uint32_t kept = 0;
                        S c0 = cdf_inv_sd(r.centre, r.inv_sd, bb[0]);
                        static_for<CB>([&](auto k) {
                            const S c1 = cdf_inv_sd(r.centre, r.inv_sd, bb[k + 1]);
                            kept |= (c1 - c0) * mor >= S(0.00001f) ? 1u << k : 0u;
                            c0 = c1;
                        });
                        static_for<3>([&](auto c) { odd_bins[c] |= (odd >> c) & 1u ? kept : 0u; });
                        odd_nan |= kept ? odd >> 3 : 0u;
                    }
                }
                S c0 = 0;
                bool have = false;
                static_for<CB / kBinGroup>([&](auto group) {
                    constexpr int k0 = group * kBinGroup;
                    // bins past the chunk's end are empty (bb repeats), so a group needs no bound
                    if (__builtin_amdgcn_ballot_w64(hi > bb[k0] && lo < bb[k0 + kBinGroup]) == 0) {
                        have = false;
                        return;
                    }
                    if (!have)
                        c0 = cdf_inv_sd(r.centre, r.inv_sd, bb[k0]);
                    have = true;
                    static_for<kBinGroup>([&](auto q) {
                        constexpr int k = k0 + q;
                        const S c1 = cdf_inv_sd(r.centre, r.inv_sd, bb[k + 1]);
                        const S mass = (c1 - c0) * mor;
                        c0 = c1;
                        const S m = mass >= S(0.00001f) ? mass : S(0); // NaN is not kept
                        bins[k][0] = dfma(g.rgb[0], m, bins[k][0]);
                        bins[k][1] = dfma(g.rgb[1], m, bins[k][1]);
                        bins[k][2] = dfma(g.rgb[2], m, bins[k][2]);
                        bins[k][3] += m;
                    });
                });
            }
            cw.store(cand);
        }
    }
    if (ODD && __builtin_amdgcn_ballot_w64((odd_bins[0] | odd_bins[1] | odd_bins[2]) != 0) != 0) {
        static_for<CB>([&](auto k) {
            static_for<3>([&](auto c) {
                const S v = (odd_nan >> c) & 1u ? S(__builtin_nan("")) : S(__builtin_huge_val());
                bins[k][c] = (odd_bins[c] >> k) & 1u ? v : bins[k][c];
            });
        });
    }
}

template <class S, int TW, int TH, int CB>
__global__ __launch_bounds__(TW* TH, sizeof(S) == 4 ? 2 : 1) void k_march_forward(MarchData<S> md, DevCamera<S> cam, MarchControl ctl, S* __restrict__ framebuffer,
    S* __restrict__ remaining, Replay<S> rp)
{
    constexpr int NT = TW * TH;
    constexpr int NCH = (kBins + CB - 1) / CB;
    __shared__ Staged<S> s_g[NT];
    __shared__ Reach1d s_win[NT];
    __shared__ uint64_t s_cand[NT / 64][2][kCandWords];
    __shared__ float s_axis[4];
    __shared__ SectionSmem<S, NT> s_sec;
    if (md.n_pairs && *md.n_pairs == 0)
        return; // no visible Gaussian: the framebuffer stays as the caller cleared it
    const int tile = xcd_tile_m(blockIdx.x, md.n_tiles);
    const int px = (tile % cam.grid_x) * TW + int(threadIdx.x) % TW;
    const int py = (tile / cam.grid_x) * TH + int(threadIdx.x) / TW;
    const bool inside = px < cam.width && py < cam.height;
    S o[3] = { cam.pos[0], cam.pos[1], cam.pos[2] };
    S d[3];
    pixel_ray(cam, inside ? px : 0, inside ? py : 0, d);
    const uint32_t first = md.ranges[2 * tile], last = md.ranges[2 * tile + 1];
    const Candidates cand = clear_candidates(s_cand[threadIdx.x / 64]);
    TileList<S, NT> tl { s_g, s_win, md, first, last, tile_axis<S>(d, inside, s_axis), last };
    const bool by_cand = sections_by_candidates(md, first, last);
    S C0 = 0, C1 = 0, C2 = 0, T = 1, start = 0;
    bool done = !inside;
    int steps = 0;
    SectionList<S, kSections, NT> sec = section_list<S, NT>(s_sec);
    while (true) {
        sec.reset(start);
        build_sections<S, NT>(sec, tl, done, inside, o, d, ctl, by_cand, cand);
        // border range of this large step
        BorderWalk<S, kSections> walk;
        walk.begin(sec);
        const S b_first = walk.prev;
        S b_last = b_first;
        {
            BorderWalk<S, kSections> w2 = walk;
            for (int k = 0; k < kBins; ++k)
                b_last = w2.next(sec);
        }
        bool stopped = done || sec.size == 0;
        // this step's replay record, when the store keeps it
        S* rec = steps < rp.steps ? rp.data + (int64_t(tile) * rp.steps + steps) * replay_record_elems<NT>() : nullptr;
        if (rec)
            rec[int64_t(NT) * (4 * kBins + kBorders) + threadIdx.x] = stopped ? S(0) : S(1);
        for (int ch = 0; ch < NCH; ++ch) {
            const int kk = min(CB, kBins - ch * CB);
            S bb[CB + 1];
            bb[0] = walk.prev;
#pragma unroll
            for (int k = 1; k <= CB; ++k)
                bb[k] = (k <= kk) ? walk.next(sec) : bb[k - 1];
            S bins[CB][4];
            fill_chunk<true, S, NT, CB>(bins, bb, stopped, tl, inside, o, d, b_first, b_last, cand);
            if (rec) {
                S* rb = rec + (int64_t(ch * CB) * NT + threadIdx.x) * 4;
                S* rd = rec + int64_t(NT) * 4 * kBins + int64_t(ch * CB) * NT + threadIdx.x;
                static_for<CB>([&](auto k) {
                    if (k < kk) {
                        store4(rb + int64_t(k) * NT * 4, detached(bins[k][0]), detached(bins[k][1]), detached(bins[k][2]), detached(bins[k][3]));
                        rd[int64_t(k) * NT] = bb[k];
                    }
                });
                if (ch == NCH - 1)
                    rd[int64_t(kk) * NT] = bb[CB];
            }
            // blend, branch-free (branches around the bins cost copies of them):
            // a stopped pixel takes nothing more, bins past the chunk's end are empty
            static_for<CB>([&](auto k) {
                C0 = stopped ? C0 : C0 + bins[k][0] * T;
                C1 = stopped ? C1 : C1 + bins[k][1] * T;
                C2 = stopped ? C2 : C2 + bins[k][2] * T;
                T = stopped ? T : T * dexp(-bins[k][3]);
                stopped = stopped || T < S(1. / 255.);
            });
        }
        ++steps;
        done = done || sec.size == 0 || T < S(1.f / 255.f) || (ctl.max_large_steps > 0 && steps >= ctl.max_large_steps);
        if (__syncthreads_count(!done) == 0)
            break;
        start = b_last;
    }
    if (rp.tile_steps && threadIdx.x == 0)
        rp.tile_steps[tile] = uint32_t(steps);
    if (!inside)
        return;
    const int64_t p = int64_t(py) * cam.width + px;
    const int64_t plane = int64_t(cam.width) * cam.height;
    framebuffer[p] = C0 + T * cam.bg[0];
    framebuffer[plane + p] = C1 + T * cam.bg[1];
    framebuffer[2 * plane + p] = C2 + T * cam.bg[2];
    remaining[p] = T;
}

// The reference's debug modes (vol_marcher_forward.cu:443-484), forward only:
//  Bins   one large step; the pixel shows (r m + g m + b m + m) * max_depth of
//         bin debug_bin (as unsigned, clamped to the last bin), green for an
//         empty bin, magenta for NaN, red for a negative sum; T = 0;
//  Depth  T *= exp(-m) over every bin (no early stop within a step), colour
//         max(end(), previous) / max_depth with end() the section list's end
//         (+inf unless the list filled up).
// A pixel that has stopped keeps taking part in its tile's later large steps
// as in the reference's block loop: its pass 1 is skipped, so its section
// list is empty and its Depth colour becomes +inf / max_depth.
template <class S, int TW, int TH, int CB>
__global__ __launch_bounds__(TW* TH) void k_march_forward_debug(MarchData<S> md, DevCamera<S> cam, MarchControl ctl,
    S* __restrict__ framebuffer, S* __restrict__ remaining)
{
    constexpr int NT = TW * TH;
    constexpr int NCH = (kBins + CB - 1) / CB;
    __shared__ Staged<S> s_g[NT];
    __shared__ Reach1d s_win[NT];
    __shared__ uint64_t s_cand[NT / 64][2][kCandWords];
    __shared__ float s_axis[4];
    __shared__ SectionSmem<S, NT> s_sec;
    if (md.n_pairs && *md.n_pairs == 0)
        return; // no visible Gaussian: the framebuffer stays as the caller cleared it
    const int tile = xcd_tile_m(blockIdx.x, md.n_tiles);
    const int px = (tile % cam.grid_x) * TW + int(threadIdx.x) % TW;
    const int py = (tile / cam.grid_x) * TH + int(threadIdx.x) / TW;
    const bool inside = px < cam.width && py < cam.height;
    S o[3] = { cam.pos[0], cam.pos[1], cam.pos[2] };
    S d[3];
    pixel_ray(cam, inside ? px : 0, inside ? py : 0, d);
    const uint32_t first = md.ranges[2 * tile], last = md.ranges[2 * tile + 1];
    const Candidates cand = clear_candidates(s_cand[threadIdx.x / 64]);
    TileList<S, NT> tl { s_g, s_win, md, first, last, tile_axis<S>(d, inside, s_axis), last };
    const bool by_cand = sections_by_candidates(md, first, last);
    const bool bins_mode = ctl.render_mode == 1;
    const int target = int(min(unsigned(ctl.debug_bin), unsigned(kBins - 1)));
    const S max_depth = S(ctl.max_depth);
    S C0 = 0, C1 = 0, C2 = 0, T = 1, start = 0, distance = 0;
    bool done = !inside;
    int steps = 0;
    SectionList<S, kSections, NT> sec = section_list<S, NT>(s_sec);
    while (true) {
        sec.reset(start);
        build_sections<S, NT>(sec, tl, done, inside, o, d, ctl, by_cand, cand);
        BorderWalk<S, kSections> walk;
        walk.begin(sec);
        const S b_first = walk.prev;
        S b_last = b_first;
        {
            BorderWalk<S, kSections> w2 = walk;
            for (int k = 0; k < kBins; ++k)
                b_last = w2.next(sec);
        }
        S bin_sum = 0;
        for (int ch = 0; ch < NCH; ++ch) {
            const int kk = min(CB, kBins - ch * CB);
            S bb[CB + 1];
            bb[0] = walk.prev;
#pragma unroll
            for (int k = 1; k <= CB; ++k)
                bb[k] = (k <= kk) ? walk.next(sec) : bb[k - 1];
            if (bins_mode && (target < ch * CB || target >= ch * CB + kk))
                continue; // only the chunk holding the shown bin
            S bins[CB][4];
            fill_chunk<true, S, NT, CB>(bins, bb, done, tl, inside, o, d, b_first, b_last, cand);
#pragma unroll
            for (int k = 0; k < CB; ++k) {
                if (k < kk) {
                    if (bins_mode) {
                        if (ch * CB + k == target)
                            bin_sum = ((bins[k][0] + bins[k][1]) + bins[k][2]) + bins[k][3];
                    } else {
                        T *= dexp(-bins[k][3]);
                    }
                }
            }
        }
        // every pixel of the tile takes the mode's blend, stopped or not (the reference's block loop)
        if (bins_mode) {
            S c[3] = { bin_sum * max_depth, bin_sum * max_depth, bin_sum * max_depth };
            if (bin_sum == S(0)) {
                c[0] = 0;
                c[1] = 1;
                c[2] = 0;
            }
            if (bin_sum != bin_sum) {
                c[0] = 1;
                c[1] = 0;
                c[2] = S(0.5);
            }
            if (bin_sum < S(0)) {
                c[0] = 1;
                c[1] = 0;
                c[2] = 0;
            }
            C0 = c[0];
            C1 = c[1];
            C2 = c[2];
            T = 0;
        } else {
            distance = dmax(sec.end_, distance);
            C0 = C1 = C2 = distance / max_depth;
        }
        ++steps;
        done = done || sec.size == 0 || T < S(1.f / 255.f) || (ctl.max_large_steps > 0 && steps >= ctl.max_large_steps);
        if (__syncthreads_count(!done) == 0)
            break;
        start = b_last;
    }
    if (!inside)
        return;
    const int64_t p = int64_t(py) * cam.width + px;
    const int64_t plane = int64_t(cam.width) * cam.height;
    framebuffer[p] = C0 + T * cam.bg[0];
    framebuffer[plane + p] = C1 + T * cam.bg[1];
    framebuffer[2 * plane + p] = C2 + T * cam.bg[2];
    remaining[p] = T;
}

template <class S>
__device__ __forceinline__ S wave_total(S v)
{
    return wave_sum_to_last(v);
}

// Blend adjoint of one chunk (grad/math.h:529-557), front to back from the
// running transmittance T and remaining colour Cr: bin k's gradient is
// dL/d(rgb mass) = Tk[k] dL/dC and dL/d(mass) = Gk[k].  Bins past the chunk
// end or after the pixel stopped get zero, and borders that make them empty.
template <class S, int CB>
__device__ __forceinline__ void blend_adjoint(const S (&bins)[CB][4], S (&bb)[CB + 1], int kk, bool& stopped, S& T, S* Cr, S Tf, S gT,
    const S* gC, S (&Tk)[CB], S (&Gk)[CB])
{
#pragma unroll
    for (int k = 0; k < CB; ++k) {
        Tk[k] = 0;
        Gk[k] = 0;
        if (k < kk && !stopped) {
            const S tk = dexp(-bins[k][3]);
            const S inv_tk = dmin(S(255), S(1) / tk);
            Cr[0] = (Cr[0] - bins[k][0]) * inv_tk;
            Cr[1] = (Cr[1] - bins[k][1]) * inv_tk;
            Cr[2] = (Cr[2] - bins[k][2]) * inv_tk;
            const S g_tk = Tf * inv_tk * gT + ((gC[0] * Cr[0] + gC[1] * Cr[1]) + gC[2] * Cr[2]) * T;
            Tk[k] = T;
            Gk[k] = -g_tk * tk;
            T *= tk;
            if (T < S(1. / 255.))
                stopped = true;
        } else {
            bb[k + 1] = bb[k];
        }
    }
}

// Pass 3: the adjoint of one chunk's deposit for every Gaussian of the tile
// (grad/math.h:559-620), summed over the wave's pixels into 13 atomics per
// Gaussian (mass 1, rgb 3, means 3, inverse covariance 6).  Per bin the
// gradient of the bin's mass is Tk (dL/dC . rgb) + Gk; the rgb gradient is
// dL/dC times the sum of Tk mass, and the centre and inverse-sd gradients
// collect the cdf derivatives at both borders of every bin.  Entries, groups of
// bins and kept bins are fill_chunk's up to the pixel's stop, past which its
// bins are empty: a pixel adds to the Gaussians it took mass from and to no
// other, also where its gradient or a colour is infinite or NaN.  RECORD: no
// deposit pass has visited the chunk's entries, so this one records which are
// the wave's candidates.
template <bool RECORD, class S, int NT, int CB>
__device__ __forceinline__ void adjoint_chunk(TileList<S, NT>& tl, const Candidates& cand, bool active, bool inside, const S* o, const S* d,
    const S (&bb)[CB + 1], S b_first, S b_last, const S (&Tk)[CB], const S (&Gk)[CB], const S* gC, S* __restrict__ render_grads)
{
    const uint32_t end = __syncthreads_count(active) == 0 ? tl.first : tl.last;
    const float inf = __builtin_inff();
    const float wlo = wave_min(active ? float(bb[0]) : inf), whi = wave_max(active ? float(bb[CB]) : -inf);
    for (uint32_t base = tl.first; base < end; base += NT) {
        tl.stage(base, o);
        const int cnt = int(min<uint32_t>(NT, tl.last - base));
        for (int j0 = 0; j0 < cnt; j0 += 64) {
            uint64_t word = entries_in(tl.s_win, j0, cnt, wlo, whi);
            if (word == 0)
                continue;
            CandidateWord cw(cand, base - tl.first + uint32_t(j0));
            for (word &= ~cw.rejected; word != 0; word &= word - 1) {
                const int j = __builtin_ctzll(word);
                const Staged<S>& g = tl.s_g[j0 + j];
                RayGauss<S> r;
                const bool pass = ray_gaussian(g, o, d, &r) && active;
                if (RECORD)
                    cw.visited(j, inside, r.mor);
                if (__builtin_amdgcn_ballot_w64(pass && r.centre + r.far > bb[0] && r.centre - r.far < bb[CB]) == 0)
                    continue;
                const bool need = deposits_in(r, pass, b_first, b_last, bb[0], bb[CB]);
                const S lo = need ? r.centre - r.far : S(inf), hi = need ? r.centre + r.far : S(-inf);
                const S mor = need ? r.mor : S(0);
                const S gcr = dfma(gC[2], g.rgb[2], dfma(gC[1], g.rgb[1], gC[0] * g.rgb[0]));
                S c0 = 0, p0 = 0, q0 = 0;
                S s_d = 0, s_tm = 0, s_c = 0, s_i = 0;
                bool have = false, contrib = false;
                static_for<CB / kBinGroup>([&](auto group) {
                    constexpr int k0 = group * kBinGroup;
                    if (__builtin_amdgcn_ballot_w64(hi > bb[k0] && lo < bb[k0 + kBinGroup]) == 0) {
                        have = false;
                        return;
                    }
                    if (!have)
                        cdf_grad_step(r.centre, r.inv_sd, bb[k0], &c0, &p0, &q0);
                    have = true;
                    static_for<kBinGroup>([&](auto bin) {
                        constexpr int k = k0 + bin;
                        S c1, p1, q1;
                        cdf_grad_step(r.centre, r.inv_sd, bb[k + 1], &c1, &p1, &q1);
                        const S delta = c1 - c0;
                        // the bin's mass max(0, m) is kept from 1e-5 on (NaN is not)
                        const bool kept = delta * mor >= S(0.00001f);
                        contrib = contrib || kept;
                        const S tk = kept ? Tk[k] : S(0);
                        const S g_m = kept ? dfma(Tk[k], gcr, Gk[k]) : S(0);
                        s_tm = dfma(tk, delta, s_tm);
                        s_d = dfma(g_m, delta, s_d);
                        s_c = dfma(g_m, p1 - p0, s_c);
                        s_i = dfma(g_m, q1 - q0, s_i);
                        c0 = c1;
                        p0 = p1;
                        q0 = q1;
                    });
                });
                if (__builtin_amdgcn_ballot_w64(contrib) == 0)
                    continue;
                S gr[13];
#pragma unroll
                for (int q = 0; q < 13; ++q)
                    gr[q] = 0;
                if (contrib) {
                    S fp, fq;
                    cdf_grad_scale(r.inv_sd, &fp, &fq);
                    // d L / d mass on the ray = s_d; weight = mor / mass
                    gr[0] = fast_div(s_d * mor, g.mass);
                    s_tm *= mor;
                    gr[1] = gC[0] * s_tm;
                    gr[2] = gC[1] * s_tm;
                    gr[3] = gC[2] * s_tm;
                    // d cdf / d centre = -inv_sd pdf; d cdf / d var = -z pdf / (2 var)
                    const S g_centre = -(s_c * mor) * fp;
                    const S g_var = -(s_i * mor) * fq * (S(0.5) * r.inv_sd * r.inv_sd);
                    intersect_ray_grad(g.mu, g.A, o, d, r.centre, s_d * mor, g_centre, g_var, gr + 4, gr + 7);
                }
                S* dst = render_grads + int64_t(g.id) * 13;
                if constexpr (sizeof(S) == 4) {
                    // two transposing reductions: lane 8m holds values kSum8Order[m] and 8 + kSum8Order[m]
                    const float ta = wave_sum8(gr[0], gr[1], gr[2], gr[3], gr[4], gr[5], gr[6], gr[7]);
                    const float tb = wave_sum8(gr[8], gr[9], gr[10], gr[11], gr[12], 0.f, 0.f, 0.f);
                    const unsigned ln = lane_id();
                    if ((ln & 7u) == 0) {
                        const int q = kSum8Order[ln >> 3];
                        unsafeAtomicAdd(dst + q, ta);
                        if (q < 5)
                            unsafeAtomicAdd(dst + 8 + q, tb);
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < 13; ++q)
                        gr[q] = wave_total(gr[q]);
                    if (lane_id() == 63) {
#pragma unroll
                        for (int q = 0; q < 13; ++q)
                            unsafeAtomicAdd(dst + q, gr[q]);
                    }
                }
            }
            if (RECORD)
                cw.store(cand);
        }
    }
}

// per-pixel state of the backward: dL/dC, the remaining colour C - T_final bg,
// T_final and dL/dT_final . bg
template <class S>
struct PixelAdjoint {
    S gC[3], Cr[3], Tf, gT;
};

template <class S>
__device__ __forceinline__ PixelAdjoint<S> load_pixel_adjoint(const DevCamera<S>& cam, bool inside, int px, int py, const S* framebuffer,
    const S* remaining, const S* grad_fb)
{
    PixelAdjoint<S> a { { 0, 0, 0 }, { 0, 0, 0 }, 1, 0 };
    if (inside) {
        const int64_t p = int64_t(py) * cam.width + px;
        const int64_t plane = int64_t(cam.width) * cam.height;
        a.Tf = remaining[p];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            a.gC[c] = grad_fb[c * plane + p];
            a.Cr[c] = framebuffer[c * plane + p] - a.Tf * cam.bg[c];
        }
    }
    a.gT = (a.gC[0] * cam.bg[0] + a.gC[1] * cam.bg[1]) + a.gC[2] * cam.bg[2];
    return a;
}

// backward replay, vol_marcher_backward.cu:126-318: sections and bins
// recomputed per large step.  With a replay store, the tiles whose block the
// store kept whole are left to k_march_backward_stored.
template <class S, int TW, int TH, int CB>
__global__ __launch_bounds__(TW* TH) void k_march_backward(MarchData<S> md, DevCamera<S> cam, MarchControl ctl, const S* __restrict__ framebuffer,
    const S* __restrict__ remaining, const S* __restrict__ grad_fb, S* __restrict__ render_grads, Replay<S> rp)
{
    constexpr int NT = TW * TH;
    constexpr int NCH = (kBins + CB - 1) / CB;
    __shared__ Staged<S> s_g[NT];
    __shared__ Reach1d s_win[NT];
    __shared__ uint64_t s_cand[NT / 64][2][kCandWords];
    __shared__ float s_axis[4];
    __shared__ SectionSmem<S, NT> s_sec;
    const int tile = xcd_tile_m(blockIdx.x, md.n_tiles);
    if (rp.tile_steps && rp.tile_steps[tile] <= uint32_t(rp.steps))
        return;
    const int px = (tile % cam.grid_x) * TW + int(threadIdx.x) % TW;
    const int py = (tile / cam.grid_x) * TH + int(threadIdx.x) / TW;
    const bool inside = px < cam.width && py < cam.height;
    S o[3] = { cam.pos[0], cam.pos[1], cam.pos[2] };
    S d[3];
    pixel_ray(cam, inside ? px : 0, inside ? py : 0, d);
    const uint32_t first = md.ranges[2 * tile], last = md.ranges[2 * tile + 1];
    const Candidates cand = clear_candidates(s_cand[threadIdx.x / 64]);
    TileList<S, NT> tl { s_g, s_win, md, first, last, tile_axis<S>(d, inside, s_axis), last };
    const bool by_cand = sections_by_candidates(md, first, last);
    PixelAdjoint<S> pa = load_pixel_adjoint(cam, inside, px, py, framebuffer, remaining, grad_fb);
    S T = 1, start = 0;
    bool done = !inside;
    int steps = 0;
    SectionList<S, kSections, NT> sec = section_list<S, NT>(s_sec);
    while (true) {
        sec.reset(start);
        build_sections<S, NT>(sec, tl, done, inside, o, d, ctl, by_cand, cand);
        BorderWalk<S, kSections> walk;
        walk.begin(sec);
        const S b_first = walk.prev;
        S b_last = b_first;
        {
            BorderWalk<S, kSections> w2 = walk;
            for (int k = 0; k < kBins; ++k)
                b_last = w2.next(sec);
        }
        bool stopped = done || sec.size == 0;
        for (int ch = 0; ch < NCH; ++ch) {
            const int kk = min(CB, kBins - ch * CB);
            S bb[CB + 1];
            bb[0] = walk.prev;
#pragma unroll
            for (int k = 1; k <= CB; ++k)
                bb[k] = (k <= kk) ? walk.next(sec) : bb[k - 1];
            S Tk[CB], Gk[CB];
            const bool active = !stopped;
            {
                S bins[CB][4];
                // pass 2 (identical to the forward)
                fill_chunk<false, S, NT, CB>(bins, bb, stopped, tl, inside, o, d, b_first, b_last, cand);
                blend_adjoint<S, CB>(bins, bb, kk, stopped, T, pa.Cr, pa.Tf, pa.gT, pa.gC, Tk, Gk);
            }
            adjoint_chunk<false, S, NT, CB>(tl, cand, active, inside, o, d, bb, b_first, b_last, Tk, Gk, pa.gC, render_grads);
        }
        ++steps;
        done = done || sec.size == 0 || T < S(1.f / 255.f) || (ctl.max_large_steps > 0 && steps >= ctl.max_large_steps);
        if (__syncthreads_count(!done) == 0)
            break;
        start = b_last;
    }
}

// The backward of the tiles the replay store kept whole: per large step the
// forward's bins and borders are read back instead of recomputed, so only the
// adjoint walks remain.  The forward and the recomputing backward hold the
// same bins (the per-bin accumulation order over Gaussians does not depend on
// the chunking), and the block takes the forward's number of large steps.
template <class S, int TW, int TH, int CB>
__global__ __launch_bounds__(TW* TH) void k_march_backward_stored(MarchData<S> md, DevCamera<S> cam, const S* __restrict__ framebuffer,
    const S* __restrict__ remaining, const S* __restrict__ grad_fb, S* __restrict__ render_grads, Replay<S> rp)
{
    constexpr int NT = TW * TH;
    constexpr int NCH = (kBins + CB - 1) / CB;
    __shared__ Staged<S> s_g[NT];
    __shared__ Reach1d s_win[NT];
    __shared__ uint64_t s_cand[NT / 64][2][kCandWords];
    __shared__ float s_axis[4];
    const int tile = xcd_tile_m(blockIdx.x, md.n_tiles);
    const uint32_t n_steps = rp.tile_steps[tile];
    if (n_steps > uint32_t(rp.steps))
        return; // recomputed by k_march_backward
    const int px = (tile % cam.grid_x) * TW + int(threadIdx.x) % TW;
    const int py = (tile / cam.grid_x) * TH + int(threadIdx.x) / TW;
    const bool inside = px < cam.width && py < cam.height;
    S o[3] = { cam.pos[0], cam.pos[1], cam.pos[2] };
    S d[3];
    pixel_ray(cam, inside ? px : 0, inside ? py : 0, d);
    const uint32_t first = md.ranges[2 * tile], last = md.ranges[2 * tile + 1];
    const Candidates cand = clear_candidates(s_cand[threadIdx.x / 64]);
    TileList<S, NT> tl { s_g, s_win, md, first, last, tile_axis<S>(d, inside, s_axis), last };
    PixelAdjoint<S> pa = load_pixel_adjoint(cam, inside, px, py, framebuffer, remaining, grad_fb);
    S T = 1;
    for (uint32_t step = 0; step < n_steps; ++step) {
        const S* rec = rp.data + (int64_t(tile) * rp.steps + step) * replay_record_elems<NT>();
        const S* rd = rec + int64_t(NT) * 4 * kBins + threadIdx.x;
        bool stopped = rd[int64_t(NT) * kBorders] == S(0);
        const S b_first = rd[0];
        const S b_last = rd[int64_t(kBins) * NT];
        for (int ch = 0; ch < NCH; ++ch) {
            const int kk = min(CB, kBins - ch * CB);
            S bb[CB + 1];
#pragma unroll
            for (int k = 0; k <= CB; ++k)
                bb[k] = rd[int64_t(ch * CB + min(k, kk)) * NT];
            S Tk[CB], Gk[CB];
            const bool active = !stopped;
            if (active) {
                S bins[CB][4];
                const S* rb = rec + (int64_t(ch * CB) * NT + threadIdx.x) * 4;
#pragma unroll
                for (int k = 0; k < CB; ++k) {
                    if (k < kk)
                        load4(rb + int64_t(k) * NT * 4, bins[k]);
                    else
                        bins[k][0] = bins[k][1] = bins[k][2] = bins[k][3] = 0;
                }
                blend_adjoint<S, CB>(bins, bb, kk, stopped, T, pa.Cr, pa.Tf, pa.gT, pa.gC, Tk, Gk);
            } else {
#pragma unroll
                for (int k = 0; k < CB; ++k)
                    Tk[k] = Gk[k] = 0;
            }
            adjoint_chunk<true, S, NT, CB>(tl, cand, active, inside, o, d, bb, b_first, b_last, Tk, Gk, pa.gC, render_grads);
        }
    }
}

// per-Gaussian adjoint of the preprocess, vol_marcher_backward.cu:321-384
template <class S>
__global__ __launch_bounds__(kPreThreads) void k_march_preprocess_backward(int64_t n, MarchArgs<S> a, DevCamera<S> cam,
    const uint32_t* __restrict__ tiles, const S* __restrict__ inv_cov, const uint8_t* __restrict__ clamped, const S* __restrict__ rg,
    S* __restrict__ g_means, S* __restrict__ g_scales, S* __restrict__ g_rot, S* __restrict__ g_opacity, S* __restrict__ g_sh)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const S* r = rg + i * 13;
    S* gsh = g_sh + i * a.sh_coeffs * 3;
    for (int c = 0; c < 3; ++c)
        g_means[3 * i + c] = r[4 + c];
    if (tiles[i] == 0) {
        for (int c = 0; c < 3; ++c)
            g_scales[3 * i + c] = 0;
        for (int c = 0; c < 4; ++c)
            g_rot[4 * i + c] = 0;
        g_opacity[i] = 0;
        for (int k = 0; k < a.sh_coeffs * 3; ++k)
            gsh[k] = 0;
        return;
    }
    const S mu[3] = { a.means[3 * i], a.means[3 * i + 1], a.means[3 * i + 2] };
    const S w = a.opacity[i];
    const S m = a.scale_multiplier;
    const S s[3] = { a.scales[3 * i] * m, a.scales[3 * i + 1] * m, a.scales[3 * i + 2] * m };
    const S q[4] = { a.rotations[4 * i], a.rotations[4 * i + 1], a.rotations[4 * i + 2], a.rotations[4 * i + 3] };
    const S delta[3] = { mu[0] - cam.pos[0], mu[1] - cam.pos[1], mu[2] - cam.pos[2] };
    const S dist = length3(delta);
    S cov[6];
    compute_cov(s, q, cov);
    const S aa = div_rn(S(kFilterSD) * cam.tan_fovx * S(2), S(cam.width));
    const S f = dist * aa;
    S W[3][3];
    for (int rr = 0; rr < 3; ++rr)
        for (int c = 0; c < 3; ++c)
            W[rr][c] = cam.view[4 * c + rr];
    S c2[3];
    affine_cut(cov, W, c2);
    const S dir[3] = { delta[0] / dist, delta[1] / dist, delta[2] / dist };
    // colour: SH coefficients beyond those stored read as 1 here, as the
    // reference binding pads them for the backward (python_bindings/vol_marcher.cu:177)
    const S gr[3] = { clamped[3 * i] ? r[1] : S(0), clamped[3 * i + 1] ? r[2] : S(0), clamped[3 * i + 2] ? r[3] : S(0) };
    S Y[16], dY[16][3];
    sh_basis(a.sh_degree, dir, Y);
    sh_basis_grad(a.sh_degree, dir, dY);
    const S* c = a.sh + i * a.sh_coeffs * 3;
    const int kact = (a.sh_degree + 1) * (a.sh_degree + 1);
    S g_dir[3] = { 0, 0, 0 };
    for (int k = 0; k < 16; ++k) {
        if (k >= kact)
            break;
        const bool stored = k < a.sh_coeffs;
        const S c0 = stored ? c[3 * k] : S(1), c1 = stored ? c[3 * k + 1] : S(1), c2v = stored ? c[3 * k + 2] : S(1);
        if (stored) {
            gsh[3 * k + 0] = Y[k] * gr[0];
            gsh[3 * k + 1] = Y[k] * gr[1];
            gsh[3 * k + 2] = Y[k] * gr[2];
        }
        const S dc = c0 * gr[0] + c1 * gr[1] + c2v * gr[2];
        g_dir[0] += dY[k][0] * dc;
        g_dir[1] += dY[k][1] * dc;
        g_dir[2] += dY[k][2] * dc;
    }
    for (int k = kact; k < a.sh_coeffs; ++k)
        gsh[3 * k] = gsh[3 * k + 1] = gsh[3 * k + 2] = 0;
    S g_mu[3] = { g_dir[0] / dist, g_dir[1] / dist, g_dir[2] / dist };
    S g_dist = -dot3(g_dir, delta) / (dist * dist);
    S g_covf[6];
    const S* A = inv_cov + 6 * i;
    sym3_inverse_grad(A, r + 7, g_covf);
    const S g_mass = r[0];
    const S det2 = c2[0] * c2[2] - c2[1] * c2[1];
    const S sq = sqrt_rn(det2);
    const S g_w = g_mass * (S(2 * kPi) * sq);
    const S fm = g_mass * w * S(2 * kPi) / (S(2) * sq);
    const S g_c2[3] = { fm * c2[2], fm * (S(-2) * c2[1]), fm * c2[0] };
    S g_cov[6], g_Wm[3][3];
    affine_cut_grad(cov, W, g_c2, g_cov, g_Wm, false);
    for (int k = 0; k < 6; ++k)
        g_cov[k] += g_covf[k];
    const S g_f2 = g_covf[0] + g_covf[3] + g_covf[5];
    g_dist += g_f2 * S(2) * f * aa;
    S g_s[3], g_q[4];
    compute_cov_grad(s, q, g_cov, g_s, g_q);
    for (int k = 0; k < 3; ++k) {
        g_mu[k] += g_dist * delta[k] / dist;
        g_means[3 * i + k] += g_mu[k];
        g_scales[3 * i + k] = g_s[k] * m;
    }
    for (int k = 0; k < 4; ++k)
        g_rot[4 * i + k] = g_q[k];
    g_opacity[i] = g_w;
}

template <class S>
MarchArgs<S> make_args(const dgmr_gaussians* g)
{
    MarchArgs<S> a;
    a.means = static_cast<const S*>(g->means);
    a.scales = static_cast<const S*>(g->scales);
    a.rotations = static_cast<const S*>(g->rotations);
    a.opacity = static_cast<const S*>(g->opacity);
    a.sh = static_cast<const S*>(g->sh);
    a.sh_coeffs = g->sh_coeffs;
    a.sh_degree = g->sh_degree;
    a.scale_multiplier = S(g->scale_multiplier);
    return a;
}

MarchControl make_control(const dgmr_march_options* opt)
{
    MarchControl c {};
    if (opt) {
        c.max_large_steps = opt->max_large_steps;
        c.n_frozen = std::min(8, std::max(0, opt->n_frozen));
        for (int k = 0; k < c.n_frozen; ++k)
            for (int j = 0; j < 3; ++j)
                c.frozen[k][j] = opt->frozen[k][j];
        c.bins_per_chunk = opt->bins_per_chunk;
        c.render_mode = opt->render_mode;
        c.debug_bin = opt->debug_render_bin;
        c.max_depth = opt->max_depth > 0 ? opt->max_depth : 20.0;
    }
    else {
        c.max_depth = 20.0;
    }
    return c;
}

template <class S, int TW, int TH>
void launch_march(bool backward, const MarchData<S>& md, const DevCamera<S>& dc, const MarchControl& ctl, S* fb, S* T, const S* gfb, S* rg,
    const Replay<S>& rp, hipStream_t st)
{
    const dim3 grid(md.n_tiles), block(TW * TH);
    // float: 32 bins in registers per pass (two waves per SIMD) unless
    // bins_per_chunk asks for 16 (three waves per SIMD, more passes): 200k
    // Gaussians at 1024^2 take 16.8 / 19.5 ms forward, 11.2 / 12.8 ms read
    // back from a replay store and 26.0 / 32.5 ms recomputed
    if constexpr (sizeof(S) == 4) {
        const bool chunk16 = ctl.bins_per_chunk == 16;
        if (!backward && ctl.render_mode == 0) {
            if (chunk16)
                k_march_forward<S, TW, TH, 16><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, rp);
            else
                k_march_forward<S, TW, TH, 32><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, rp);
            return;
        }
        if (backward) {
            if (rp.steps > 0) {
                if (chunk16)
                    k_march_backward_stored<S, TW, TH, 16><<<grid, block, 0, st>>>(md, dc, fb, T, gfb, rg, rp);
                else
                    k_march_backward_stored<S, TW, TH, 32><<<grid, block, 0, st>>>(md, dc, fb, T, gfb, rg, rp);
            }
            if (chunk16)
                k_march_backward<S, TW, TH, 16><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, gfb, rg, rp);
            else
                k_march_backward<S, TW, TH, 32><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, gfb, rg, rp);
            return;
        }
    }
    constexpr int CB = sizeof(S) == 4 ? 32 : 16;
    if (!backward && ctl.render_mode != 0)
        k_march_forward_debug<S, TW, TH, 16><<<grid, block, 0, st>>>(md, dc, ctl, fb, T);
    else if (!backward)
        k_march_forward<S, TW, TH, CB><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, rp);
    else {
        if (rp.steps > 0)
            k_march_backward_stored<S, TW, TH, CB><<<grid, block, 0, st>>>(md, dc, fb, T, gfb, rg, rp);
        k_march_backward<S, TW, TH, CB><<<grid, block, 0, st>>>(md, dc, ctl, fb, T, gfb, rg, rp);
    }
}

template <class S>
void dispatch_march(const dgmr_tiling& t, bool backward, const MarchData<S>& md, const DevCamera<S>& dc, const MarchControl& ctl, S* fb, S* T,
    const S* gfb, S* rg, const Replay<S>& rp, hipStream_t st)
{
    if (t.tile_w == 16)
        launch_march<S, 16, 16>(backward, md, dc, ctl, fb, T, gfb, rg, rp, st);
    else if (t.tile_w == 8)
        launch_march<S, 8, 8>(backward, md, dc, ctl, fb, T, gfb, rg, rp, st);
    else
        launch_march<S, 32, 8>(backward, md, dc, ctl, fb, T, gfb, rg, rp, st);
}

// bytes of a replay store keeping `steps` large steps of every tile: the
// per-tile step counts (padded to 256 bytes), then the records
int64_t replay_bytes(int64_t n_tiles, int threads_per_tile, int steps, size_t scalar)
{
    const int64_t head = (n_tiles * 4 + 255) / 256 * 256;
    return head + n_tiles * int64_t(steps) * int64_t(threads_per_tile) * (4 * kBins + kBorders + 1) * int64_t(scalar);
}

// the store the options name, checked against this frame's size
template <class S>
int make_replay(const dgmr_march_options* opt, const dgmr_tiling& t, int64_t n_tiles, Replay<S>* rp)
{
    *rp = Replay<S> { nullptr, nullptr, 0 };
    if (!opt || !opt->replay)
        return DGMR_OK;
    DGMR_ARG_CHECK(opt->replay_steps >= 1, "dgmr_march: replay_steps must be >= 1 with a replay store");
    DGMR_ARG_CHECK(opt->replay_bytes >= size_t(replay_bytes(n_tiles, t.tile_w * t.tile_h, opt->replay_steps, sizeof(S))),
        "dgmr_march: replay store smaller than dgmr_march_replay_size");
    DGMR_ARG_CHECK(reinterpret_cast<uintptr_t>(opt->replay) % 256 == 0, "dgmr_march: replay store must be 256-byte aligned");
    const int64_t head = (n_tiles * 4 + 255) / 256 * 256;
    rp->tile_steps = static_cast<uint32_t*>(opt->replay);
    rp->data = reinterpret_cast<S*>(static_cast<char*>(opt->replay) + head);
    rp->steps = opt->replay_steps;
    return DGMR_OK;
}

template <class S>
int march_forward_t(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, const dgmr_march_options* opt,
    dgmr_march_geometry* geom, dgmr_binning* bins, void* framebuffer, void* remaining, void* workspace, size_t workspace_bytes,
    dgmr_stats* stats, hipStream_t st)
{
    const int64_t n = g->n;
    const DevCamera<S> dc = make_dev_camera<S>(*cam, *tiling);
    const int64_t n_tiles = int64_t(dc.grid_x) * dc.grid_y;
    const int64_t plane = int64_t(cam->width) * cam->height;
    if (stats)
        stats->n_pairs = 0;
    Replay<S> rp;
    if (const int rc = make_replay<S>(opt, *tiling, n_tiles, &rp); rc != DGMR_OK)
        return rc;
    // an empty visible set leaves an all-zero image (vol_marcher_forward.cu:193-195 with
    // the binding's zero-initialised framebuffer, python_bindings/vol_marcher.cu:83)
    DGMR_HIP_CHECK(hipMemsetAsync(framebuffer, 0, size_t(3 * plane) * sizeof(S), st));
    if (n == 0) {
        DGMR_HIP_CHECK(hipMemsetAsync(bins->ranges, 0, size_t(n_tiles) * 2 * sizeof(uint32_t), st));
        return DGMR_OK;
    }
    const MarchArgs<S> a = make_args<S>(g);
    uint32_t *dkeys, *dids;
    binning_key_buffers(workspace, n, false, &dkeys, &dids);
    {
        StageScope sc("march.preprocess", st, double(n) * sizeof(S) * (14.0 + 3.0 * g->sh_coeffs + 16.0));
        k_march_preprocess<S><<<unsigned(ceil_div64(n, kPreThreads)), kPreThreads, 0, st>>>(n, a, dc, geom->rects, geom->tiles_touched,
            static_cast<S*>(geom->xy), static_cast<S*>(geom->depths), static_cast<S*>(geom->rgb), geom->rgb_clamped,
            static_cast<S*>(geom->inverse_filtered_cov3d), static_cast<S*>(geom->filtered_masses), dkeys, dids);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    Carver cv(workspace, workspace_bytes);
    PendingCount pending;
    const int rc = bin_gaussians(n, geom->rects, geom->tiles_touched, geom->xy, sizeof(S) == 8, false, false, dc.grid_x, dc.grid_y, dc.tile_w, dc.tile_h, bins, cv,
        &pending, st, nullptr);
    if (rc != DGMR_OK)
        return rc;
    // with no pair at all the kernel leaves the caller's zero framebuffer
    // untouched (vol_marcher_forward.cu:193-195)
    MarchData<S> md { bins->ranges, bins->point_list, a.means, static_cast<const S*>(geom->inverse_filtered_cov3d), static_cast<const S*>(geom->rgb),
        static_cast<const S*>(geom->filtered_masses), static_cast<const S*>(geom->depths), int(n_tiles), pending.device };
    const MarchControl ctl = make_control(opt);
    if (ctl.render_mode != 0) {
        // the debug modes keep nothing: every tile is recomputed by the backward
        if (rp.tile_steps)
            DGMR_HIP_CHECK(hipMemsetAsync(rp.tile_steps, 0xff, size_t(n_tiles) * 4, st));
        rp = Replay<S> { nullptr, nullptr, 0 };
    }
    {
        StageScope sc("march.render_forward", st);
        pending.add_stage(sc.slot, 4.0 + 15.0 * sizeof(S), double(plane) * 4.0 * sizeof(S));
        dispatch_march<S>(*tiling, false, md, dc, ctl, static_cast<S*>(framebuffer), static_cast<S*>(remaining), nullptr, nullptr, rp, st);
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

template <class S>
int march_backward_t(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, const dgmr_march_options* opt,
    const dgmr_march_geometry* geom, const dgmr_binning* bins, int64_t n_pairs, const void* framebuffer, const void* remaining,
    const void* grad_fb, void* render_grads, void* g_means, void* g_scales, void* g_rot, void* g_opacity, void* g_sh, hipStream_t st)
{
    const int64_t n = g->n;
    if (n == 0)
        return DGMR_OK;
    const DevCamera<S> dc = make_dev_camera<S>(*cam, *tiling);
    const int64_t n_tiles = int64_t(dc.grid_x) * dc.grid_y;
    const MarchArgs<S> a = make_args<S>(g);
    Replay<S> rp;
    if (const int rc = make_replay<S>(opt, *tiling, n_tiles, &rp); rc != DGMR_OK)
        return rc;
    DGMR_HIP_CHECK(hipMemsetAsync(render_grads, 0, size_t(n) * 13 * sizeof(S), st));
    if (n_pairs > 0) {
        MarchData<S> md { bins->ranges, bins->point_list, a.means, static_cast<const S*>(geom->inverse_filtered_cov3d),
            static_cast<const S*>(geom->rgb), static_cast<const S*>(geom->filtered_masses), static_cast<const S*>(geom->depths), int(n_tiles),
            nullptr }; // the host knows n_pairs > 0: no device count
        StageScope sc("march.render_backward", st, double(n_pairs) * (4.0 + 15.0 * sizeof(S)));
        dispatch_march<S>(*tiling, true, md, dc, make_control(opt), const_cast<S*>(static_cast<const S*>(framebuffer)),
            const_cast<S*>(static_cast<const S*>(remaining)), static_cast<const S*>(grad_fb), static_cast<S*>(render_grads), rp, st);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    StageScope sc("march.preprocess_backward", st, double(n) * sizeof(S) * (2.0 * (14.0 + 3.0 * g->sh_coeffs) + 19.0));
    k_march_preprocess_backward<S><<<unsigned(ceil_div64(n, kPreThreads)), kPreThreads, 0, st>>>(n, a, dc, geom->tiles_touched,
        static_cast<const S*>(geom->inverse_filtered_cov3d), geom->rgb_clamped, static_cast<const S*>(render_grads), static_cast<S*>(g_means),
        static_cast<S*>(g_scales), static_cast<S*>(g_rot), static_cast<S*>(g_opacity), static_cast<S*>(g_sh));
    DGMR_HIP_CHECK(hipGetLastError());
    return DGMR_OK;
}

} // namespace
} // namespace dgmr

using namespace dgmr;

extern "C" {

int dgmr_march_forward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, const dgmr_march_options* opt,
    dgmr_march_geometry* geom, dgmr_binning* bins, void* framebuffer, void* remaining_transparency, void* workspace, size_t workspace_bytes,
    dgmr_stats* stats, dgmr_stream stream)
{
    DGMR_ARG_CHECK(g && cam && geom && bins && framebuffer && remaining_transparency && workspace, "dgmr_march_forward: null argument");
    DGMR_ARG_CHECK(g->dtype == DGMR_F32 || g->dtype == DGMR_F64, "dgmr_march_forward: dtype must be float32 or float64");
    DGMR_ARG_CHECK(valid_tiling(tiling) && tiling->cull == 0, "dgmr_march_forward: bad tiling (the marcher bins whole rectangles)");
    DGMR_ARG_CHECK(g->n >= 0 && g->n < (int64_t(1) << 31), "dgmr_march_forward: bad Gaussian count");
    DGMR_ARG_CHECK(g->sh_coeffs >= 1 && g->sh_coeffs <= 16 && g->sh_degree >= 0 && g->sh_degree <= 3, "dgmr_march_forward: bad SH layout");
    DGMR_ARG_CHECK(g->activation == DGMR_ACT_NONE, "dgmr_march_forward: the marcher takes activated parameters");
    DGMR_ARG_CHECK(valid_image(cam->width, cam->height), "dgmr_march_forward: bad image size");
    DGMR_ARG_CHECK(workspace_bytes >= splat_workspace_bytes(g->n, bins->pair_capacity), "dgmr_march_forward: workspace too small");
    DGMR_ARG_CHECK(!opt || (opt->render_mode >= 0 && opt->render_mode <= 2), "dgmr_march_forward: render_mode must be 0 (full), 1 (bins) or 2 (depth)");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (g->dtype == DGMR_F32)
        return march_forward_t<float>(g, cam, tiling, opt, geom, bins, framebuffer, remaining_transparency, workspace, workspace_bytes, stats, st);
    return march_forward_t<double>(g, cam, tiling, opt, geom, bins, framebuffer, remaining_transparency, workspace, workspace_bytes, stats, st);
}

int dgmr_march_replay_size(int32_t width, int32_t height, const dgmr_tiling* tiling, int32_t replay_steps, int32_t dtype, size_t* bytes)
{
    DGMR_ARG_CHECK(bytes && valid_tiling(tiling), "dgmr_march_replay_size: bad argument");
    DGMR_ARG_CHECK(valid_image(width, height), "dgmr_march_replay_size: bad image size");
    DGMR_ARG_CHECK(replay_steps >= 1 && replay_steps <= 1024, "dgmr_march_replay_size: replay_steps must be in [1, 1024]");
    DGMR_ARG_CHECK(dtype == DGMR_F32 || dtype == DGMR_F64, "dgmr_march_replay_size: dtype must be float32 or float64");
    const int64_t n_tiles = int64_t((width + tiling->tile_w - 1) / tiling->tile_w) * ((height + tiling->tile_h - 1) / tiling->tile_h);
    *bytes = size_t(replay_bytes(n_tiles, tiling->tile_w * tiling->tile_h, replay_steps, dtype == DGMR_F32 ? 4 : 8));
    return DGMR_OK;
}

int dgmr_march_backward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, const dgmr_march_options* opt,
    const dgmr_march_geometry* geom, const dgmr_binning* bins, int64_t n_pairs, const void* framebuffer, const void* remaining_transparency,
    const void* grad_framebuffer, void* render_grads, void* grad_means, void* grad_scales, void* grad_rotations, void* grad_opacity, void* grad_sh,
    dgmr_stream stream)
{
    DGMR_ARG_CHECK(g && cam && geom && bins && framebuffer && remaining_transparency && grad_framebuffer && render_grads,
        "dgmr_march_backward: null argument");
    DGMR_ARG_CHECK(grad_means && grad_scales && grad_rotations && grad_opacity && grad_sh, "dgmr_march_backward: null gradient output");
    DGMR_ARG_CHECK(g->dtype == DGMR_F32 || g->dtype == DGMR_F64, "dgmr_march_backward: dtype must be float32 or float64");
    DGMR_ARG_CHECK(valid_tiling(tiling) && tiling->cull == 0, "dgmr_march_backward: bad tiling (the marcher bins whole rectangles)");
    DGMR_ARG_CHECK(g->sh_coeffs >= 1 && g->sh_coeffs <= 16 && g->sh_degree >= 0 && g->sh_degree <= 3, "dgmr_march_backward: bad SH layout");
    DGMR_ARG_CHECK(g->activation == DGMR_ACT_NONE, "dgmr_march_backward: the marcher takes activated parameters");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (g->dtype == DGMR_F32)
        return march_backward_t<float>(g, cam, tiling, opt, geom, bins, n_pairs, framebuffer, remaining_transparency, grad_framebuffer, render_grads,
            grad_means, grad_scales, grad_rotations, grad_opacity, grad_sh, st);
    return march_backward_t<double>(g, cam, tiling, opt, geom, bins, n_pairs, framebuffer, remaining_transparency, grad_framebuffer, render_grads,
        grad_means, grad_scales, grad_rotations, grad_opacity, grad_sh, st);
}

} // extern "C"
