// SPDX-License-Identifier: GPL-3.0-or-later
// Tile splatter for gfx950: forward (reference: src/dgmr/splat_forward.cu:30-338)
// and the backward the reference does not ship.
//
// Pipeline (one stream, one 4-byte read-back for the pair count):
//   1. k_splat_preprocess   per Gaussian: EWA splat (Ots, 0.3 px^2 filter), rect,
//                           tiles touched, depth key, SH colour, conic.
//   2. radix sort of the Gaussians by depth bits (stable, ties by index)
//   3. k_gather_owners      tiles touched and tile rectangle in depth order,
//                           exclusive scan -> pair offsets
//   4. k_emit_bounds, k_emit_pairs   pair-balanced emission of (tile id, Gaussian id)
//   5. radix sort of the pairs by tile id only (stable)
//      Steps 2-5 yield exactly the order of the reference's single sort on
//      (tile << 32 | depth bits): within a tile, pairs stay in (depth bits,
//      Gaussian id) order, which is the reference's stable order.
//   6. k_tile_ranges        [first, last) per tile (binary search per tile)
//   7. k_blend_forward      per tile, LDS-staged batches of Gaussians
// A view of at most 16 384 Gaussians takes steps 2 and 3 and the bounds in one
// launch (k_bin_one); the autograd path bins deep views by a prefix of the depth
// order where that pays (k_prefix_decide, k_extend_*, k_open_*).
// Backward: k_blend_backward (front-to-back replay, transmittance recomputed,
// wave-reduced atomics) then k_splat_preprocess_backward (per Gaussian).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "device_grad.h"
#include "device_math.h"
#include "host_common.h"
#include "primitives.h"
#include "splat_device.h"

namespace dgmr {

namespace {

constexpr int kPreThreads = 256;
// depth sorts of at least this many keys compact the visible entries first
constexpr int64_t kCompactMin = int64_t(4) << 20;

__global__ __launch_bounds__(kPreThreads) void k_splat_preprocess(int64_t n, SplatParams p, DevCamera<float> cam, SplatOut out)
{
    // SH rows are read straight from global memory: the 12 row loads of a wave
    // cover one contiguous span that stays in cache, and keeping LDS free
    // keeps the occupancy that hides the gather latency
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        preprocess_gaussian(i, i, p, p.sh + i * p.sh_coeffs * 3, cam, out);
}

} // namespace

// Emission of (tile, Gaussian) pairs balanced over pairs: block b writes pairs
// [b * kEmitPairs, (b + 1) * kEmitPairs) of the depth-ordered pair list.  Its
// first owner and an upper bound of its last come from k_emit_bounds; the
// owners in between (culled Gaussians carry the largest depth key, so the
// owners of a block's pairs are contiguous and each owns at least one pair)
// are staged in LDS with their tile rectangle, and every thread writes
// kEmitPer consecutive pairs.  A window wider than the LDS stage (more than
// kEmitWindow owners in one block's pairs, or zero-pair Gaussians among
// visible ones) takes a per-pair search instead.
// views: per-view (grid_x, grid_y, first global tile, -) when ids span several
// views of n_per_view Gaussians each; null for a single view.
constexpr int kEmitThreads = 256;
// pairs per thread: 8, or 16 from kEmitLarge pairs up (the per-thread search
// and setup spread over more pairs: 434M pairs 1.13 -> 1.06 ms; at 15M, with
// half the blocks, 16 was slower, 0.042 against 0.032 ms)
constexpr int kEmitPerSmall = 8, kEmitPerLarge = 16;
static_assert((kEmitThreads & (kEmitThreads - 1)) == 0 && (kEmitPerSmall & (kEmitPerSmall - 1)) == 0 && (kEmitPerLarge & (kEmitPerLarge - 1)) == 0,
    "an emission block's pairs: a power of two");
constexpr int64_t kEmitLarge = int64_t(48) << 20;
constexpr int kEmitWindow = 2048; // owners a block stages in LDS (more take the per-pair search)

// First owners of the emission blocks: bounds[b] is the Gaussian (position
// in depth order) that owns pair b << block_shift, for every block that emits,
// and bounds[n_blocks] owns the last emitted pair.  Position k owns pairs
// [offsets[k], offsets[k + 1]) and writes the entries whose pair falls in its
// range, so each entry is written exactly once and no block searches.
__device__ __forceinline__ void emit_bounds_of(uint32_t k, uint64_t lo, uint64_t next, uint64_t total, uint32_t capacity, int block_shift,
    uint32_t* __restrict__ bounds)
{
    const uint64_t R = min(total, uint64_t(capacity)); // pairs past the capacity are not emitted
    const uint64_t hi = min(next, R);
    if (lo >= hi)
        return;
    const uint64_t up = (uint64_t(1) << block_shift) - 1;
    for (uint64_t b = (lo + up) >> block_shift; (b << block_shift) < hi; ++b)
        bounds[b] = k;
    if (R - 1 < hi)
        bounds[(R + up) >> block_shift] = k;
}
__global__ void k_emit_bounds(int64_t n, const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ n_pairs, uint32_t capacity,
    const uint32_t* __restrict__ n_emit, int block_shift, uint32_t* __restrict__ bounds)
{
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n)
        return;
    const uint64_t total = *n_pairs;
    emit_bounds_of(uint32_t(k), offsets[k], k + 1 < n ? uint64_t(offsets[k + 1]) : total, total, min(*n_emit, capacity), block_shift, bounds);
}

// tile rectangle of Gaussian id: first tile and (grid_x << 16 | width); 0 shape when it has no tiles
template <class S>
__device__ __forceinline__ void owner_rect(uint32_t id, const int32_t* __restrict__ rects, const uint32_t* __restrict__ tiles,
    const S* __restrict__ xy, int grid_x, int grid_y, int tile_w, int tile_h, const int4* __restrict__ views, int64_t n_per_view,
    uint32_t* start, uint32_t* shape)
{
    *start = 0;
    *shape = 0;
    if (tiles[id] == 0)
        return;
    int gx = grid_x, gy = grid_y, tbase = 0;
    if (views) {
        const int4 v = views[id / uint32_t(n_per_view)]; // ids < 2^32: a 32-bit division
        gx = v.x;
        gy = v.y;
        tbase = v.z;
    }
    int a, b, c, d;
    get_rect(xy[2 * id], xy[2 * id + 1], rects[2 * id], rects[2 * id + 1], gx, gy, tile_w, tile_h, &a, &b, &c, &d);
    // sort keys are view-local tile ids (the view comes back through the id)
    (void)tbase;
    *start = uint32_t(b) * uint32_t(gx) + uint32_t(a);
    *shape = (uint32_t(gx) << 16) | uint32_t(c - a);
}

// What k_prefix_decide sums up, per cell of the image: sixteenths of a pixel, pairs
struct DecideSums {
    unsigned long long alpha[64], rest[64];
    uint32_t blocks;
};
// Tile rectangles by position of the depth order for the lists' extension (null: not
// wanted): (row << 16 | column) of the first tile, (rows << 16 | columns)
struct PrefixRects {
    uint32_t* origin;
    uint32_t* size;
    DecideSums* sums; // to be cleared
};

// Per position j of the depth order: the pair count of Gaussian ids[j] (for
// the scan) and its tile rectangle (for the emission).  The random reads of
// per-Gaussian data happen here, in a streaming kernel, so the emission reads
// its owners' rectangles as contiguous runs; with the preprocess's packed bin
// rectangle that is one 8-byte read per Gaussian.
template <class S, bool RECTS>
__global__ __launch_bounds__(256) void k_gather_owners(int64_t n, const uint32_t* __restrict__ n_sorted, const uint32_t* __restrict__ ids,
    const uint2* __restrict__ bin_rects,
    const int32_t* __restrict__ rects, const uint32_t* __restrict__ tiles, const S* __restrict__ xy, int grid_x, int grid_y, int tile_w,
    int tile_h, const int4* __restrict__ views, int64_t n_per_view, uint32_t* __restrict__ counts, uint2* __restrict__ owner_rects,
    ScanState scan, PrefixRects prefix)
{
    scan_clear(scan); // for the scan of counts that follows
    if (prefix.sums && blockIdx.x == 0) {
        if (threadIdx.x < 64)
            prefix.sums->alpha[threadIdx.x] = prefix.sums->rest[threadIdx.x] = 0;
        if (threadIdx.x == 0)
            prefix.sums->blocks = 0;
    }
    const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (j >= n)
        return;
    if (n_sorted && j >= int64_t(*n_sorted)) {
        // past the compacted (visible) entries: no pairs
        counts[j] = 0;
        owner_rects[j] = make_uint2(0u, 0u);
        return;
    }
    const uint32_t id = ids[j];
    uint32_t start, shape, count;
    if constexpr (RECTS) {
        const uint2 r = bin_rects[id];
        const uint32_t cols = r.y & 0xffffu, rows = r.y >> 16;
        const uint32_t gx = views ? uint32_t(views[id / uint32_t(n_per_view)].x) : uint32_t(grid_x);
        start = r.x;
        shape = cols * rows == 0 ? 0u : (gx << 16) | cols;
        count = cols * rows;
        if (prefix.origin) {
            const uint32_t y = start / gx;
            prefix.origin[j] = (y << 16) | (start - y * gx);
            prefix.size[j] = r.y;
        }
    } else {
        owner_rect(id, rects, tiles, xy, grid_x, grid_y, tile_w, tile_h, views, n_per_view, &start, &shape);
        count = tiles[id];
    }
    counts[j] = count;
    owner_rects[j] = make_uint2(start, shape);
}

// ------------------------------------------------------- small views' binning
// Depth sort, gather, both scans and the emission's bounds of a view of at most
// kBinOneMax Gaussians in one workgroup.  As separate launches these are 16 to
// 18 of a few microseconds each with gaps as long between them; one CU has the
// whole view in its registers and LDS.  The sort is the stable LSD radix sort
// of the large path (equal digits found by ballot, a running count per wave and
// digit), on the visible depth keys less the smallest of them: a view's depths
// span few octaves, so the bits that all keys share are not sorted.  Culled
// Gaussians (key ~0) take the key after the last and stay in order behind.
// Bound by the latency of its passes on one CU: 12.6 us at 301 Gaussians and 39
// us at 10 000, against 66 us and 75 us of the launches it replaces; at 16 384 a
// whole forward call of 256x256 pixels takes 134 us, at 16 385 with the launches
// 155.  Above kBinOneMax the keys no longer fit its registers and LDS and the launches of
// the large path fill more CUs (50 000: 12 launches in 60 us).
constexpr int kBinOneThreads = 1024;
constexpr int kBinOneItems = 16;
constexpr int kBinOneWaves = kBinOneThreads / 64;
constexpr int64_t kBinOneMax = int64_t(kBinOneThreads) * kBinOneItems;
constexpr int kBinOneRadix = 512;

struct BinOneArgs {
    int n;
    const uint32_t* keys;   // depth bits, ~0 culled
    const uint2* bin_rects;
    const uint32_t* tiles;
    uint32_t grid_x;
    uint32_t capacity;
    int block_shift;        // log2 of the pairs of an emission block
    uint32_t* ids;
    uint2* owner_rects;
    uint32_t* offsets;
    uint32_t* point_offsets; // by a second workgroup
    uint32_t* n_pairs;
    uint32_t* bounds;
};

// exclusive scan of s[0..n) in place, by the whole workgroup; returns the sum.
// A thread's share is an odd number of items, so its lanes fall on different banks.
__device__ __forceinline__ uint32_t bin_one_scan(uint32_t* s, int n, uint32_t* s_wave)
{
    const unsigned lane = lane_id(), wave = threadIdx.x / 64;
    const int per = ((n + kBinOneThreads - 1) / kBinOneThreads) | 1;
    const int first = min(int(threadIdx.x) * per, n), last = min(first + per, n);
    uint32_t sum = 0;
    for (int i = first; i < last; ++i)
        sum += s[i];
    uint32_t v = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane >= unsigned(d))
            v += o;
    }
    if (lane == 63)
        s_wave[wave] = v;
    __syncthreads();
    uint32_t run = v - sum, total = 0;
#pragma unroll
    for (unsigned w = 0; w < kBinOneWaves; ++w) {
        const uint32_t c = s_wave[w];
        run += w < wave ? c : 0u;
        total += c;
    }
    for (int i = first; i < last; ++i) {
        const uint32_t x = s[i];
        s[i] = run;
        run += x;
    }
    __syncthreads();
    return total;
}

__global__ __launch_bounds__(kBinOneThreads) void k_bin_one(BinOneArgs a)
{
    __shared__ uint32_t s_key[kBinOneMax];
    __shared__ uint16_t s_id[kBinOneMax];
    __shared__ uint16_t s_count[kBinOneWaves][kBinOneRadix]; // counts, then places: below 2^15
    __shared__ uint32_t s_wave[kBinOneWaves], s_lo[kBinOneWaves], s_hi[kBinOneWaves];
    const int n = a.n, t = int(threadIdx.x);
    const unsigned lane = lane_id(), wave = threadIdx.x / 64;
    const uint64_t lt = (uint64_t(1) << lane) - 1;
    const int rounds = (n + kBinOneThreads - 1) / kBinOneThreads;
    const int own = int(wave) * rounds * 64 + int(lane); // this lane's item of round 0
    if (blockIdx.x == 1) {
        // the second workgroup: the inclusive scan of the tile counts in id order
        for (int j = t; j < n; j += kBinOneThreads)
            s_key[j] = a.tiles[j];
        __syncthreads();
        const uint32_t all = bin_one_scan(s_key, n, s_wave);
        for (int j = t; j < n; j += kBinOneThreads)
            a.point_offsets[j] = j + 1 < n ? s_key[j + 1] : all;
        return;
    }
    uint32_t key[kBinOneItems], id[kBinOneItems]; // id: the rank in the (wave, digit) in the upper half
    uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
    for (int r = 0; r < kBinOneItems; ++r) {
        const int i = own + r * 64;
        id[r] = uint32_t(i);
        key[r] = r < rounds && i < n ? a.keys[i] : 0xffffffffu;
    }
#pragma unroll
    for (int r = 0; r < kBinOneItems; ++r) {
        if (key[r] != 0xffffffffu) {
            lo = min(lo, key[r]);
            hi = max(hi, key[r]);
        }
        if (r < rounds && own + r * 64 < n)
            s_id[own + r * 64] = uint16_t(own + r * 64); // stays when nothing is visible
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        lo = min(lo, uint32_t(__shfl_xor(int(lo), d, 64)));
        hi = max(hi, uint32_t(__shfl_xor(int(hi), d, 64)));
    }
    if (lane == 0) {
        s_lo[wave] = lo;
        s_hi[wave] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kBinOneWaves; ++w) {
        lo = min(lo, s_lo[w]);
        hi = max(hi, s_hi[w]);
    }
    lo = uniform(lo);
    hi = uniform(hi);
    const uint32_t behind = hi - lo + 1u; // the culled entries' key
    const int bits = lo <= hi ? 32 - __clz(int(behind)) : 0;
#pragma unroll
    for (int r = 0; r < kBinOneItems; ++r)
        key[r] = key[r] == 0xffffffffu ? behind : key[r] - lo;
    const auto pass = [&](int shift, auto width) {
        constexpr int W = decltype(width)::value;
        constexpr uint32_t mask = (1u << W) - 1u;
        constexpr int kWords = (1 << W) / 2; // counters, two to a word
        for (int i = t; i < kBinOneWaves * kBinOneRadix / 2; i += kBinOneThreads)
            reinterpret_cast<uint32_t*>(&s_count[0][0])[i] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBinOneItems; ++r) {
            if (r < rounds) {
                const bool valid = own + r * 64 < n;
                const uint32_t digit = (key[r] >> shift) & mask;
                const uint64_t valid_lanes = __ballot(valid);
                uint32_t peers_lo = uint32_t(valid_lanes), peers_hi = uint32_t(valid_lanes >> 32);
#pragma unroll
                for (int b = 0; b < W; ++b) {
                    const uint32_t s = uint32_t(int32_t(digit << (31 - b)) >> 31);
                    const uint64_t m = __ballot(s != 0u);
                    peers_lo &= ~(uint32_t(m) ^ s);
                    peers_hi &= ~(uint32_t(m >> 32) ^ s);
                }
                const uint64_t peers = (uint64_t(peers_hi) << 32) | peers_lo;
                // every lane reads the count before the lowest lane of its digit writes it back
                const uint32_t before = s_count[wave][digit];
                id[r] |= (before + uint32_t(__popcll(peers & lt))) << 16;
                if (valid && (peers & lt) == 0)
                    s_count[wave][digit] = uint16_t(before + uint32_t(__popcll(peers)));
                __builtin_amdgcn_wave_barrier();
            }
        }
        __syncthreads();
        {
            // thread d < kWords: the starts of digits 2d and 2d + 1 per wave,
            // exclusive over the digits (both halves of a word at once: no sum reaches 2^16)
            uint32_t c[kBinOneWaves], tot = 0;
#pragma unroll
            for (int w = 0; w < kBinOneWaves; ++w) {
                c[w] = t < kWords ? reinterpret_cast<const uint32_t*>(s_count[w])[t] : 0u;
                tot += c[w];
            }
            const uint32_t sum = (tot & 0xffffu) + (tot >> 16);
            uint32_t v = sum;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const uint32_t o = __shfl_up(v, k, 64);
                if (lane >= unsigned(k))
                    v += o;
            }
            if (lane == 63)
                s_wave[wave] = v;
            __syncthreads();
            if (t < kWords) {
                uint32_t start = v - sum;
#pragma unroll
                for (unsigned w = 0; w < kWords / 64; ++w)
                    start += w < wave ? s_wave[w] : 0u;
                start |= (start + (tot & 0xffffu)) << 16;
#pragma unroll
                for (int w = 0; w < kBinOneWaves; ++w) {
                    reinterpret_cast<uint32_t*>(s_count[w])[t] = start;
                    start += c[w];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBinOneItems; ++r) {
            if (r < rounds && own + r * 64 < n) {
                const uint32_t pos = s_count[wave][(key[r] >> shift) & mask] + (id[r] >> 16);
                s_key[pos] = key[r];
                s_id[pos] = uint16_t(id[r]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBinOneItems; ++r) {
            if (r < rounds && own + r * 64 < n) {
                key[r] = s_key[own + r * 64];
                id[r] = s_id[own + r * 64];
            }
        }
    };
    // 9-bit digits (one to three passes) up to 27 bits, 16 octaves; else four of 8
    if (bits <= 27) {
        for (int shift = 0; shift < bits; shift += 9)
            pass(shift, std::integral_constant<int, 9> {});
    } else {
        for (int shift = 0; shift < 32; shift += 8)
            pass(shift, std::integral_constant<int, 8> {});
    }
    __syncthreads(); // the keys have been read: their LDS holds the pair counts from here
    uint2 rect[kBinOneItems];
#pragma unroll
    for (int r = 0; r < kBinOneItems; ++r) {
        const int j = r * kBinOneThreads + t;
        id[r] = r < rounds && j < n ? uint32_t(s_id[j]) : 0u;
        rect[r] = r < rounds && j < n ? a.bin_rects[id[r]] : make_uint2(0u, 0u);
    }
#pragma unroll
    for (int r = 0; r < kBinOneItems; ++r) {
        const int j = r * kBinOneThreads + t;
        if (r < rounds && j < n) {
            const uint32_t cols = rect[r].y & 0xffffu, rows = rect[r].y >> 16;
            a.ids[j] = id[r];
            a.owner_rects[j] = make_uint2(rect[r].x, cols * rows == 0 ? 0u : (a.grid_x << 16) | cols);
            s_key[j] = cols * rows;
        }
    }
    __syncthreads();
    const uint32_t total = bin_one_scan(s_key, n, s_wave);
    if (t == 0)
        *a.n_pairs = total;
    for (int j = t; j < n; j += kBinOneThreads) {
        const uint32_t first = s_key[j], next = j + 1 < n ? s_key[j + 1] : total;
        a.offsets[j] = first;
        emit_bounds_of(uint32_t(j), first, next, total, a.capacity, a.block_shift, a.bounds);
    }
}

// kEmitPer consecutive pairs at a 16-byte aligned position: 32-bit keys and
// the values four to a store, 16-bit keys packed eight to a store
template <int kEmitPer>
__device__ __forceinline__ void store_run(uint32_t* keys, uint32_t* vals, const uint32_t (&kv)[kEmitPer], const uint32_t (&vv)[kEmitPer])
{
    static_assert(kEmitPer % 8 == 0, "pairs per thread: a multiple of 8");
    uint4* kd = reinterpret_cast<uint4*>(keys);
    uint4* vd = reinterpret_cast<uint4*>(vals);
#pragma unroll
    for (int j = 0; j < kEmitPer / 4; ++j) {
        kd[j] = make_uint4(kv[4 * j], kv[4 * j + 1], kv[4 * j + 2], kv[4 * j + 3]);
        vd[j] = make_uint4(vv[4 * j], vv[4 * j + 1], vv[4 * j + 2], vv[4 * j + 3]);
    }
}
template <int kEmitPer>
__device__ __forceinline__ void store_run(uint16_t* keys, uint32_t* vals, const uint32_t (&kv)[kEmitPer], const uint32_t (&vv)[kEmitPer])
{
    uint4* kd = reinterpret_cast<uint4*>(keys);
    uint4* vd = reinterpret_cast<uint4*>(vals);
#pragma unroll
    for (int j = 0; j < kEmitPer / 8; ++j)
        kd[j] = make_uint4(kv[8 * j] | (kv[8 * j + 1] << 16), kv[8 * j + 2] | (kv[8 * j + 3] << 16), kv[8 * j + 4] | (kv[8 * j + 5] << 16),
            kv[8 * j + 6] | (kv[8 * j + 7] << 16));
#pragma unroll
    for (int j = 0; j < kEmitPer / 4; ++j)
        vd[j] = make_uint4(vv[4 * j], vv[4 * j + 1], vv[4 * j + 2], vv[4 * j + 3]);
}

// Tight culling: per position j of the depth order, the pair count of
// Gaussian ids[j] (tiles its reach ellipse meets, row by row) and its record,
// copied so the emission reads its owners' records as contiguous runs.
// Entries the preprocess culled have no record: they are those past n_sorted
// (compacted sorts) or whose final sort key is culled_key.
__global__ __launch_bounds__(256) void k_gather_reach(int64_t n, const uint32_t* __restrict__ n_sorted, const uint32_t* __restrict__ keys,
    uint32_t culled_key, const uint32_t* __restrict__ ids, const ReachRec* __restrict__ reach, int tile_w, int tile_h,
    uint32_t* __restrict__ counts, ReachRec* __restrict__ owners, ScanState scan)
{
    scan_clear(scan); // for the scan of counts that follows
    const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (j >= n)
        return;
    uint4* dst = reinterpret_cast<uint4*>(owners + j);
    if ((n_sorted && j >= int64_t(*n_sorted)) || keys[j] == culled_key) {
        counts[j] = 0;
        dst[0] = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    const uint4* src = reinterpret_cast<const uint4*>(reach + ids[j]);
    const uint4 w0 = src[0], w1 = src[1];
    uint32_t count = 0;
    if (w0.y != 0u) {
        const ReachRec r { w0.x, w0.y, w0.z, __uint_as_float(w0.w), __uint_as_float(w1.x), __uint_as_float(w1.y), __uint_as_float(w1.z),
            __uint_as_float(w1.w) };
        const ReachEllipse e = reach_ellipse(r);
        const int x0 = int(r.origin & 0xffffu), y0 = int(r.origin >> 16), cols = int(r.dims & 0xffffu), rows = int(r.dims >> 16);
        for (int q = 0; q < rows; ++q) {
            const int2 c = reach_columns(e, y0 + q, x0, cols, tile_w, tile_h);
            if (c.x <= c.y)
                count += uint32_t(c.y - c.x + 1);
        }
    }
    counts[j] = count;
    dst[0] = w0;
    dst[1] = w1;
}

// the emission cursor of one owner: its tile row r (from the rectangle's
// first), that row's reached columns c, and the column offset within them
struct ReachCursor {
    ReachEllipse e;
    int x0, y0, cols, rows, gx;
    int r;
    int2 c;
};

__device__ __forceinline__ void cursor_load(ReachCursor& cu, const ReachRec* __restrict__ owners, uint32_t k, int tile_w, int tile_h)
{
    const uint4* src = reinterpret_cast<const uint4*>(owners + k);
    const uint4 w0 = src[0], w1 = src[1];
    const ReachRec r { w0.x, w0.y, w0.z, __uint_as_float(w0.w), __uint_as_float(w1.x), __uint_as_float(w1.y), __uint_as_float(w1.z),
        __uint_as_float(w1.w) };
    cu.e = reach_ellipse(r);
    cu.x0 = int(r.origin & 0xffffu);
    cu.y0 = int(r.origin >> 16);
    cu.cols = int(r.dims & 0xffffu);
    cu.rows = int(r.dims >> 16);
    cu.gx = int(r.grid_x);
    cu.r = 0;
    cu.c = reach_columns(cu.e, cu.y0, cu.x0, cu.cols, tile_w, tile_h);
}

// moves the cursor to the row holding column offset *local (from the current
// row) and returns the tile; rows past the rectangle are never entered
__device__ __forceinline__ uint32_t cursor_tile(ReachCursor& cu, uint32_t* local, int tile_w, int tile_h)
{
    while (cu.r < cu.rows) {
        const uint32_t w = cu.c.x <= cu.c.y ? uint32_t(cu.c.y - cu.c.x + 1) : 0u;
        if (*local < w)
            break;
        *local -= w;
        ++cu.r;
        if (cu.r < cu.rows)
            cu.c = reach_columns(cu.e, cu.y0 + cu.r, cu.x0, cu.cols, tile_w, tile_h);
    }
    return uint32_t(cu.y0 + cu.r) * uint32_t(cu.gx) + uint32_t(cu.c.x) + *local;
}

// Tight-culling emission: the same block layout as k_emit_pairs; each thread
// writes kEmitPer consecutive pairs, walking its owners' reached rows.
template <class KeyT, int kEmitPer>
__global__ __launch_bounds__(kEmitThreads) void k_emit_reach(const uint32_t* __restrict__ n_pairs, uint32_t capacity,
    const uint32_t* __restrict__ sorted_ids, const uint32_t* __restrict__ bounds, const uint32_t* __restrict__ offsets,
    const ReachRec* __restrict__ owners, int tile_w, int tile_h, KeyT* __restrict__ keys_out, uint32_t* __restrict__ vals_out)
{
    constexpr int kEmitPairs = kEmitThreads * kEmitPer;
    __shared__ uint32_t s_off[kEmitWindow];
    const uint32_t R = min(*n_pairs, capacity);
    const uint32_t first = blockIdx.x * uint32_t(kEmitPairs);
    if (first >= R)
        return;
    const uint32_t end = min(R, first + uint32_t(kEmitPairs));
    const uint32_t g_lo = bounds[blockIdx.x], g_hi = bounds[blockIdx.x + 1];
    const uint32_t window = g_hi - g_lo + 1;
    const bool staged = window <= uint32_t(kEmitWindow);
    if (staged) {
        for (uint32_t k = threadIdx.x; k < window; k += kEmitThreads)
            s_off[k] = offsets[g_lo + k];
        __syncthreads();
    }
    // start of owner g_lo + k's pairs; past the window: no end within this block
    auto off = [&](uint32_t k) -> uint32_t {
        if (k >= window)
            return 0xffffffffu;
        return staged ? s_off[k] : offsets[g_lo + k];
    };
    const uint32_t p0 = first + threadIdx.x * kEmitPer;
    if (p0 >= end)
        return;
    uint32_t lo = 0, hi = window - 1; // owner of p0: last k with off(k) <= p0
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (off(mid) <= p0)
            lo = mid;
        else
            hi = mid - 1;
    }
    uint32_t k = lo;
    uint32_t next = off(k + 1);
    uint32_t local = p0 - off(k);
    ReachCursor cu;
    cursor_load(cu, owners, g_lo + k, tile_w, tile_h);
    uint32_t id = sorted_ids[g_lo + k];
    uint32_t kv[kEmitPer], vv[kEmitPer];
#pragma unroll
    for (int q = 0; q < kEmitPer; ++q) {
        const uint32_t p = p0 + q;
        if (p >= end) {
            kv[q] = vv[q] = 0u;
            continue;
        }
        if (p >= next) {
            do {
                ++k;
                next = off(k + 1);
            } while (p >= next);
            cursor_load(cu, owners, g_lo + k, tile_w, tile_h);
            id = sorted_ids[g_lo + k];
            local = 0;
        }
        kv[q] = cursor_tile(cu, &local, tile_w, tile_h);
        vv[q] = id;
        ++local;
    }
    const bool aligned = ((reinterpret_cast<uintptr_t>(keys_out) | reinterpret_cast<uintptr_t>(vals_out)) & 15u) == 0;
    if (aligned && p0 + kEmitPer <= end) {
        store_run(keys_out + p0, vals_out + p0, kv, vv);
    } else {
#pragma unroll
        for (int q = 0; q < kEmitPer; ++q)
            if (p0 + q < end) {
                keys_out[p0 + q] = KeyT(kv[q]);
                vals_out[p0 + q] = vv[q];
            }
    }
}

template <class KeyT, int kEmitPer>
__global__ __launch_bounds__(kEmitThreads) void k_emit_pairs(int64_t n, const uint32_t* __restrict__ n_pairs, uint32_t capacity,
    const uint32_t* __restrict__ sorted_ids, const uint32_t* __restrict__ bounds, const uint32_t* __restrict__ offsets,
    const uint2* __restrict__ owner_rects, KeyT* __restrict__ keys_out, uint32_t* __restrict__ vals_out)
{
    constexpr int kEmitPairs = kEmitThreads * kEmitPer;
    __shared__ uint32_t s_off[kEmitWindow], s_id[kEmitWindow], s_start[kEmitWindow], s_shape[kEmitWindow];
    const uint32_t R = min(*n_pairs, capacity); // pairs past the capacity are not written
    const uint32_t first = blockIdx.x * uint32_t(kEmitPairs);
    if (first >= R)
        return;
    const uint32_t end = min(R, first + uint32_t(kEmitPairs));
    // owners of the block's first pair and of the next block's first pair (or
    // of the last pair): the owners of this block's pairs lie in between
    const uint32_t g_lo = bounds[blockIdx.x], g_hi = bounds[blockIdx.x + 1];
    const uint32_t window = g_hi - g_lo + 1;
    if (window <= uint32_t(kEmitWindow)) {
        for (uint32_t k = threadIdx.x; k < window; k += kEmitThreads) {
            const uint2 r = owner_rects[g_lo + k];
            s_off[k] = offsets[g_lo + k];
            s_id[k] = sorted_ids[g_lo + k];
            s_start[k] = r.x;
            s_shape[k] = r.y;
        }
        __syncthreads();
        const uint32_t p0 = first + threadIdx.x * kEmitPer;
        if (p0 >= end)
            return;
        // owner of p0: last k with s_off[k] <= p0
        uint32_t lo = 0, hi = window - 1;
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (s_off[mid] <= p0)
                lo = mid;
            else
                hi = mid - 1;
        }
        uint32_t k = lo;
        uint32_t next = k + 1 < window ? s_off[k + 1] : 0xffffffffu;
        uint32_t shape = s_shape[k], local = p0 - s_off[k];
        uint32_t w = shape & 0xffffu;
        uint32_t ty = local / w, tx = local - ty * w;
        uint32_t kv[kEmitPer], vv[kEmitPer];
#pragma unroll
        for (int q = 0; q < kEmitPer; ++q) {
            const uint32_t p = p0 + q;
            if (p >= next) {
                do {
                    ++k;
                    next = k + 1 < window ? s_off[k + 1] : 0xffffffffu;
                } while (p >= next);
                shape = s_shape[k];
                w = shape & 0xffffu;
                tx = 0;
                ty = 0;
            }
            kv[q] = s_start[k] + ty * (shape >> 16) + tx;
            vv[q] = s_id[k];
            if (++tx == w) {
                tx = 0;
                ++ty;
            }
        }
        const bool aligned = ((reinterpret_cast<uintptr_t>(keys_out) | reinterpret_cast<uintptr_t>(vals_out)) & 15u) == 0;
        if (aligned && p0 + kEmitPer <= end) {
            // 16-byte aligned: p0 is a multiple of kEmitPer
            store_run(keys_out + p0, vals_out + p0, kv, vv);
        } else {
#pragma unroll
            for (int q = 0; q < kEmitPer; ++q)
                if (p0 + q < end) {
                    keys_out[p0 + q] = KeyT(kv[q]);
                    vals_out[p0 + q] = vv[q];
                }
        }
    } else {
        for (uint32_t p = first + threadIdx.x; p < end; p += kEmitThreads) {
            uint32_t lo = g_lo, hi = g_hi;
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo + 1) >> 1);
                if (offsets[mid] <= p)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const uint32_t id = sorted_ids[lo];
            const uint2 r = owner_rects[lo];
            const uint32_t start = r.x, shape = r.y;
            const uint32_t local = p - offsets[lo];
            const uint32_t w = shape & 0xffffu;
            const uint32_t ty = local / w, tx = local - ty * w;
            keys_out[p] = KeyT(start + ty * (shape >> 16) + tx);
            vals_out[p] = id;
        }
    }
}

// What prefix binning (below) notes of the tiles whose lists it leaves open: a
// bit per tile, words of 32 along the rows; whether there is one (0 or 1); the
// groups of 8 x 8 tiles that hold one; and for the extension the positions of
// the depth order that it looks at (0 when there is none) and the pairs it makes
struct OpenTiles {
    uint32_t* tiles; // null: whole lists
    int row_words;
    int64_t words;
    uint32_t* any;
    uint32_t* positions;
    uint32_t* rest;
    uint32_t* groups;      // their number, then the groups
    uint32_t* group_noted; // [groups]
};

// [first, last) of every tile by binary search over the sorted pairs: one
// thread per tile, every tile written (an empty tile gets (0, 0)).
// The sorted order is (view-local tile, view, depth); a pair's view is
// val / n_per_view, and val >= v * n_per_view exactly when its view is >= v.
// So both ends of tile t of view v are partition points of a predicate that
// is monotone along the array: "key > t, or key == t and val >= bound".  With
// one view the bound is 0 and the two ends are the lower bounds of t and t + 1.
// The two searches of a thread run interleaved.
template <class KeyT>
__global__ __launch_bounds__(256) void k_tile_ranges(const KeyT* __restrict__ keys, const uint32_t* __restrict__ vals,
    const uint32_t* __restrict__ n_pairs, uint32_t capacity, const int4* __restrict__ views, int n_views, int64_t n_per_view, int64_t n_tiles,
    uint32_t* __restrict__ ranges, OpenTiles open)
{
    const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= n_tiles)
        return;
    if (open.tiles) {
        // for the blend and the extension of the lists (no more words or groups than tiles)
        open.group_noted[g] = 0;
        if (g < open.words)
            open.tiles[g] = 0;
        if (g == 0)
            *open.any = *open.rest = open.groups[0] = 0;
    }
    const uint32_t R = min(*n_pairs, capacity);
    uint32_t t0 = uint32_t(g), t1 = uint32_t(g) + 1;
    uint64_t b0 = 0, b1 = 0;
    if (views) {
        int lo = 0, hi = n_views - 1; // last view whose first tile is <= g
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (int64_t(views[mid].z) <= g)
                lo = mid;
            else
                hi = mid - 1;
        }
        t0 = t1 = uint32_t(g - views[lo].z);
        b0 = uint64_t(lo) * uint64_t(n_per_view);
        b1 = b0 + uint64_t(n_per_view);
    }
    uint32_t lo0 = 0, hi0 = R, lo1 = 0, hi1 = R;
    while (lo0 < hi0 || lo1 < hi1) {
        const uint32_t m0 = lo0 + (hi0 - lo0) / 2, m1 = lo1 + (hi1 - lo1) / 2;
        const bool a0 = lo0 < hi0, a1 = lo1 < hi1;
        const uint32_t k0 = a0 ? uint32_t(keys[m0]) : 0u, k1 = a1 ? uint32_t(keys[m1]) : 0u;
        const uint32_t v0 = a0 && views ? vals[m0] : 0u, v1 = a1 && views ? vals[m1] : 0u;
        const bool after0 = k0 > t0 || (k0 == t0 && uint64_t(v0) >= b0);
        const bool after1 = k1 > t1 || (k1 == t1 && uint64_t(v1) >= b1);
        if (a0) {
            if (after0)
                hi0 = m0;
            else
                lo0 = m0 + 1;
        }
        if (a1) {
            if (after1)
                hi1 = m1;
            else
                lo1 = m1 + 1;
        }
    }
    // an empty tile holds (0, 0), as the reference's zero-filled ranges
    ranges[2 * g] = lo0 < lo1 ? lo0 : 0u;
    ranges[2 * g + 1] = lo0 < lo1 ? lo1 : 0u;
}

// prefix binning (below): the first pass notes which waves' lists ended with an
// open pixel and keeps those waves' pixels as they stand; the second (again)
// goes on with them where their lists were left
struct PrefixPass {
    uint32_t* units;      // [tiles * waves per tile]: open; null: whole lists
    OpenTiles open;
    const uint32_t* done; // per open tile the entries that the first pass walked
    const uint32_t* n_pairs;
    const uint32_t* n_emit;
    uint32_t pairs;
    int split;            // waves per tile of the first pass
    bool again;
};

// kBlendWaves independent waves per workgroup, LDS private per wave, each on one
// of a tile's SPLIT bands of TH / SPLIT rows (SPLIT waves walk the tile's list)
template <int TW, int TH, int B, int SPLIT>
__global__ __launch_bounds__(64 * kBlendWaves) void k_blend_forward(const uint32_t* __restrict__ ranges, const uint32_t* __restrict__ point_list,
    const float2* __restrict__ xy, const float4* __restrict__ conic_opacity, const float* __restrict__ rgb, int width, int height, int grid_x,
    int n_tiles, float bg0, float bg1, float bg2, float* __restrict__ framebuffer, float* __restrict__ final_T, PrefixPass prefix)
{
    __shared__ BlendSmem<B> sm_all[kBlendWaves];
    if (prefix.again && *prefix.open.any == 0)
        return;
    const int wave = int(uniform(threadIdx.x / 64));
    const int unit = xcd_tile(blockIdx.x, gridDim.x) * kBlendWaves + wave;
    const int tile = unit / SPLIT, part = unit % SPLIT;
    if (tile >= n_tiles)
        return;
    if (prefix.again && uniform(prefix.units[tile * prefix.split + part % prefix.split]) == 0)
        return;
    BlendSmem<B>& sm = sm_all[wave];
    uint32_t first = uniform(ranges[2 * tile]);
    const uint32_t last = uniform(ranges[2 * tile + 1]);
    if (prefix.again)
        first = min(first + uniform(prefix.done[tile]), last);
    // whether the lists are prefixes
    const BlendResume resume { prefix.again, prefix.units && !prefix.again && *prefix.n_emit == prefix.pairs && *prefix.n_pairs > prefix.pairs };
    const bool open = blend_tile_forward<TW, TH / SPLIT, B>(sm, first, last, (tile % grid_x) * TW, (tile / grid_x) * TH + part * (TH / SPLIT),
        width, height, bg0, bg1, bg2, point_list, xy, conic_opacity, rgb, framebuffer, final_T, resume);
    if (resume.keep && lane_id() == 0) {
        prefix.units[unit] = open ? 1u : 0u;
        if (open) {
            const int tx = tile % grid_x, ty = tile / grid_x;
            const int group = ty / 8 * ((grid_x + 7) / 8) + tx / 8;
            atomicOr(&prefix.open.tiles[ty * prefix.open.row_words + tx / 32], 1u << (tx % 32));
            if (atomicExch(&prefix.open.group_noted[group], 1u) == 0)
                prefix.open.groups[1 + atomicAdd(&prefix.open.groups[0], 1u)] = uint32_t(group);
            *prefix.open.any = 1u;
        }
    }
}

// ------------------------------------------------------------ prefix binning
// A deep view's tiles saturate long before their lists end: 1M Gaussians at
// 1920x1080 make 14.9M pairs, 1 827 per tile, of which a tile walks 76 on
// average and 166 at most.  Emission and pair sort of all of them are
// bandwidth bound and were a fifth of the forward.  With prefix binning only
// the first pairs of the depth order (kPrefixPerTile per tile of the image) are
// emitted and sorted, so every tile's list is a prefix of its whole list; the
// blend notes the tiles whose list ends with a pixel still open, and the whole
// lists of these tiles are built behind the prefixes for a second blend, which
// goes on where the first one stopped.  The launches of the extension leave at
// once when no tile is open.
// Where tiles stay open prefixes cost more than they save, so a view must have
// kPrefixMin times their pairs, make 1.3M fewer (by the 16 pairs a Gaussian makes
// in an ordinary deep view) and look covered (k_prefix_decide).  Forward in us,
// prefixes / whole lists, at 1920x1080 (scales e^-3, cube of side 10 unless noted):
//   1M, opacities around 1/2      352 / 446   no tile open
//   3M, the same                  696 / 1026  3 open
//   1M, around 0.27               442 / 505   23 open
//   1M, around 0.18               562 / 539   1 004 open (whole; 544 with k_prefix_decide)
//   1M, around 0.007              1004 / 888  all open (whole; 898 with k_prefix_decide)
//   1M in a cube of side 3        610 / 698   1 838 open at its edges
//   3M in it, scales e^-4         985 / 975   618 open
constexpr int64_t kPrefixPerTile = 256;
constexpr int64_t kPrefixPairsPerGaussian = 16;
constexpr int64_t kPrefixMinSaved = 1300000;
constexpr int64_t kPrefixMin = 6;
static_assert((kPrefixMinSaved + kPrefixPerTile) / kPrefixPairsPerGaussian > kBinOneMax, "small views are binned whole");

// the first pairs that a view of n Gaussians and n_tiles tiles bins with prefix
// binning when it has kPrefixMin times as many, 0 when its whole lists are
// binned whatever it has
static int64_t prefix_pairs(int64_t n, int64_t n_tiles, int64_t pair_capacity)
{
    const int64_t pairs = kPrefixPerTile * n_tiles, expected = kPrefixPairsPerGaussian * n;
    return pair_capacity >= kPrefixMin * pairs && expected >= kPrefixMin * pairs && expected - pairs >= kPrefixMinSaved
            && pair_capacity + pairs <= int64_t(UINT32_MAX) && n_tiles <= (int64_t(1) << 22)
        ? pairs
        : 0;
}

// Whether a view's prefixes are worth while, from 4 096 Gaussians of the prefix
// and as many behind it, at equal steps of the depth order (10 us).  Per cell of
// an 8 x 8 grid of the image the first give the depth of alpha that the prefix
// lays over its pixels (a pixel is saturated at 9.2), the second the share of the
// other pairs: whole lists where more than a sixteenth of these lie in cells
// below kPrefixAlpha, which separates the scenes of the table above (no pairs at
// opacities around 0.27, a sixth of them around 0.18).  Few tiles are expected to
// be open where at most a 64th lies in cells below kFewAlpha.
constexpr int kDecideThreads = 512, kDecideBlocks = 8; // one CU alone took twice as long over its scattered loads
constexpr int kDecideSamples = kDecideThreads * kDecideBlocks;
constexpr int kCells = 8;
constexpr float kPrefixAlpha = 11.f, kFewAlpha = 12.f;
struct DecideArgs {
    int64_t n;
    const uint32_t* offsets;
    const uint32_t* n_pairs;
    uint32_t capacity, prefix;
    bool always; // the prefix whenever there are kPrefixMin times its pairs
    const uint32_t* ids;
    const uint32_t* origin;
    const uint32_t* size;
    const float4* conic_opacity;
    int grid_x, grid_y, tile_pixels;
    DecideSums* sums; // cleared by the gather
    uint32_t* n_emit;
    uint32_t* few; // whether few tiles are expected to be left open
    uint32_t* n_owners;
};

// first tile column (row) of a cell column (row): tile t lies in cell t kCells / grid
__device__ __forceinline__ int cell_edge(int cell, int grid) { return (cell * grid + kCells - 1) / kCells; }

// first position whose offset reaches v (offsets ascend), by a wave
__device__ __forceinline__ uint32_t wave_lower_bound(const uint32_t* __restrict__ offsets, uint32_t n, uint32_t v)
{
    uint32_t lo = 0, hi = n; // the answer lies in [lo, hi]
    while (lo < hi) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint32_t at = lo + lane_id() * step;
        const bool below = at < hi && offsets[at] < v;
        const uint32_t count = uint32_t(__builtin_popcountll(__builtin_amdgcn_ballot_w64(below))); // lanes in a row from 0
        if (count == 0)
            hi = lo;
        else {
            hi = min(hi, lo + count * step);
            lo = lo + (count - 1) * step + 1;
        }
    }
    return lo;
}

__global__ __launch_bounds__(kDecideThreads) void k_prefix_decide(DecideArgs a)
{
    __shared__ unsigned long long s_alpha[kCells * kCells], s_rest[kCells * kCells]; // sixteenths of a pixel; pairs
    __shared__ uint32_t s_at[2];
    const int t = int(threadIdx.x);
    const uint32_t total = *a.n_pairs, limit = min(total, a.capacity);
    const bool deep = total <= a.capacity && total >= uint64_t(kPrefixMin) * a.prefix;
    if (t < 128 && deep) {
        const uint32_t at = wave_lower_bound(a.offsets, uint32_t(a.n), t < 64 ? a.prefix : total);
        if (t % 64 == 0)
            s_at[t / 64] = at;
    }
    if (t < kCells * kCells)
        s_alpha[t] = s_rest[t] = 0;
    __syncthreads();
    const uint32_t owners = s_at[1], front = min(s_at[0], owners);
    if (!deep || a.always || front == 0 || front == owners) {
        if (t == 0 && blockIdx.x == 0) {
            *a.n_emit = deep && front < owners ? a.prefix : limit;
            *a.few = 0;
            *a.n_owners = deep ? owners : 0;
        }
        return;
    }
    const uint64_t i = uint64_t(blockIdx.x) * kDecideThreads + uint64_t(t);
    const uint32_t pos[2] = { uint32_t(i * front / kDecideSamples), front + uint32_t(i * (owners - front) / kDecideSamples) };
    const float4 c = a.conic_opacity[a.ids[pos[0]]];
    // the integral of alpha over the screen, at most its tiles' pixels, and the
    // pairs: each cell gets its share of the rectangle
    const float alpha = c.w * 6.2831853f * __builtin_amdgcn_rsqf(c.x * c.z - c.y * c.y);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t o = a.origin[pos[q]], sz = a.size[pos[q]], cols = sz & 0xffffu, rows = sz >> 16;
        const int x0 = int(o & 0xffffu), y0 = int(o >> 16), x1 = x0 + int(cols), y1 = y0 + int(rows);
        const float each = q == 0 ? fminf(alpha * __builtin_amdgcn_rcpf(float(cols) * float(rows)), float(a.tile_pixels)) : 0.f;
        for (int cy = y0 * kCells / a.grid_y; cy <= (y1 - 1) * kCells / a.grid_y; ++cy)
            for (int cx = x0 * kCells / a.grid_x; cx <= (x1 - 1) * kCells / a.grid_x; ++cx) {
                const int w = min(x1, cell_edge(cx + 1, a.grid_x)) - max(x0, cell_edge(cx, a.grid_x));
                const int h = min(y1, cell_edge(cy + 1, a.grid_y)) - max(y0, cell_edge(cy, a.grid_y));
                const float tiles = float(w) * float(h);
                if (q == 1)
                    atomicAdd(&s_rest[cy * kCells + cx], static_cast<unsigned long long>(tiles));
                else if (each > 0.f) // not for NaN
                    atomicAdd(&s_alpha[cy * kCells + cx], static_cast<unsigned long long>(each * tiles * 16.f));
            }
    }
    __syncthreads();
    if (t < 64) {
        static_assert(kCells * kCells == 64, "a lane per cell");
        atomicAdd(&a.sums->alpha[t], s_alpha[t]);
        atomicAdd(&a.sums->rest[t], s_rest[t]);
        __threadfence();
    }
    __syncthreads();
    if (t == 0)
        s_at[0] = atomicAdd(&a.sums->blocks, 1u);
    __syncthreads();
    if (s_at[0] != kDecideBlocks - 1)
        return;
    // the last workgroup decides
    if (t < 64) {
        const int x = t % kCells, y = t / kCells;
        const int tiles_x = cell_edge(x + 1, a.grid_x) - cell_edge(x, a.grid_x), tiles_y = cell_edge(y + 1, a.grid_y) - cell_edge(y, a.grid_y);
        const float pixels = float(max(tiles_x * tiles_y, 1)) * float(a.tile_pixels);
        const float depth = float(atomicAdd(&a.sums->alpha[t], 0ull)) * (1.f / 16.f) * (float(front) / float(kDecideSamples)) / pixels;
        float rest = float(atomicAdd(&a.sums->rest[t], 0ull)), open = depth < kPrefixAlpha ? rest : 0.f, thin = depth < kFewAlpha ? rest : 0.f;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            rest += __shfl_xor(rest, d);
            open += __shfl_xor(open, d);
            thin += __shfl_xor(thin, d);
        }
        if (t == 0) {
            *a.n_emit = open * 16.f <= rest ? a.prefix : limit;
            *a.few = thin * 64.f <= rest ? 1u : 0u;
            *a.n_owners = owners;
        }
    }
}

// The extension elsewhere is the binning's own emission and sort over the
// Gaussians that hold an open tile.  These, their rectangles
// shrunk to the open tiles (in place: first tile, columns), so that few open
// tiles make few pairs.  Four positions per thread: the grid costs when there is
// nothing to do.  LDS: the open tiles fit (8 192 words: 262 144 tiles and more).
constexpr int kOpenPer = 4;
constexpr int kOpenLdsWords = 8192;
template <bool LDS>
__global__ __launch_bounds__(256) void k_open_owners(OpenTiles open, int grid_x, const uint32_t* __restrict__ n_owners,
    uint32_t* __restrict__ origin, uint32_t* __restrict__ size, uint32_t* __restrict__ counts, uint32_t* __restrict__ flags, ScanState scan)
{
    extern __shared__ uint32_t s_tiles[];
    const int64_t owners = *open.any == 0 ? 0 : int64_t(*n_owners);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *open.positions = uint32_t(owners);
    if (owners == 0)
        return;
    scan_clear(scan); // for the scan of counts and flags that follows
    if (int64_t(blockIdx.x) * kOpenPer * 256 >= owners)
        return;
    if (LDS) {
        for (int i = int(threadIdx.x); i < int(open.words); i += 256)
            s_tiles[i] = open.tiles[i];
        __syncthreads();
    }
    for (int q = 0; q < kOpenPer; ++q) {
        const int64_t j = (int64_t(blockIdx.x) * kOpenPer + q) * 256 + threadIdx.x;
        if (j >= owners)
            return;
        uint32_t xa = 0xffffffffu, xb = 0, ya = 0xffffffffu, yb = 0; // the open tiles' columns and rows, ends included
        {
            // no Gaussian that owns pairs has an empty rectangle
            const uint32_t o = origin[j], sz = size[j];
            const uint32_t x0 = o & 0xffffu, y0 = o >> 16, x1 = x0 + (sz & 0xffffu) - 1, y1 = y0 + (sz >> 16) - 1;
            for (uint32_t w = x0 / 32; w <= x1 / 32; ++w) {
                const uint32_t lo = w == x0 / 32 ? x0 % 32 : 0u, hi = w == x1 / 32 ? x1 % 32 : 31u;
                const uint32_t mask = (0xffffffffu >> (31 - hi)) & (0xffffffffu << lo);
                uint32_t cols = 0;
                for (uint32_t y = y0; y <= y1; ++y) {
                    const uint32_t at = y * uint32_t(open.row_words) + w;
                    const uint32_t m = (LDS ? s_tiles[at] : open.tiles[at]) & mask;
                    cols |= m;
                    ya = m ? min(ya, y) : ya;
                    yb = m ? max(yb, y) : yb;
                }
                if (cols) {
                    xa = min(xa, 32 * w + uint32_t(__builtin_ctz(cols)));
                    xb = max(xb, 32 * w + 31u - uint32_t(__builtin_clz(cols)));
                }
            }
        }
        const uint32_t cols = xa <= xb ? xb - xa + 1 : 0u, rows = xa <= xb ? yb - ya + 1 : 0u;
        counts[j] = cols * rows;
        flags[j] = cols ? 1u : 0u;
        if (cols) {
            origin[j] = ya * uint32_t(grid_x) + xa;
            size[j] = cols;
        }
    }
}

// The owners one behind the other (the emission searches the owners of its
// pairs, and few open tiles leave few of many), and the emission blocks' first ones
__global__ __launch_bounds__(256) void k_open_bounds(OpenTiles open, const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ place,
    const uint32_t* __restrict__ start, const uint32_t* __restrict__ cols, const uint32_t* __restrict__ ids, int grid_x, uint32_t capacity,
    int block_shift, uint32_t* __restrict__ offsets_out, uint2* __restrict__ rects_out, uint32_t* __restrict__ ids_out, uint32_t* __restrict__ bounds)
{
    if (*open.any == 0)
        return;
    const uint64_t total = *open.rest;
    const int64_t n = *open.positions;
    for (int q = 0; q < kOpenPer; ++q) {
        const int64_t j = (int64_t(blockIdx.x) * kOpenPer + q) * 256 + threadIdx.x;
        if (j >= n)
            return;
        const uint32_t lo = offsets[j];
        const uint64_t next = j + 1 < n ? uint64_t(offsets[j + 1]) : total;
        if (lo >= next)
            continue;
        const uint32_t c = place[j];
        offsets_out[c] = lo;
        rects_out[c] = make_uint2(start[j], (uint32_t(grid_x) << 16) | cols[j]);
        ids_out[c] = ids[j];
        emit_bounds_of(c, lo, next, total, capacity, block_shift, bounds);
    }
}

// ranges of the open tiles in their whole lists (from entry `base` on), and the
// entries of their prefixes
template <class KeyT>
__global__ __launch_bounds__(256) void k_open_ranges(const KeyT* __restrict__ keys, uint32_t capacity, uint32_t base, OpenTiles open, int grid_x,
    int64_t n_tiles, uint32_t* __restrict__ ranges, uint32_t* __restrict__ done)
{
    const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (*open.any == 0 || g >= n_tiles)
        return;
    const int tx = int(g % grid_x), ty = int(g / grid_x);
    if (((open.tiles[ty * open.row_words + tx / 32] >> (tx % 32)) & 1u) == 0)
        return;
    const uint32_t R = min(*open.rest, capacity);
    uint32_t end[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        uint32_t lo = 0, hi = R;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (int64_t(keys[mid]) >= g + k)
                hi = mid;
            else
                lo = mid + 1;
        }
        end[k] = lo;
    }
    done[g] = ranges[2 * g + 1] - ranges[2 * g];
    ranges[2 * g] = end[0] < end[1] ? base + end[0] : 0u;
    ranges[2 * g + 1] = end[0] < end[1] ? base + end[1] : 0u;
}

// The extension where few tiles are expected to be open (three launches: 11 us
// without one, 62 us with 3 of 8 160 at 3M, where k_open_owners and the emission
// and sort take 32 and 116; all tiles open 600 us at 1M, those 200) works on groups of 8 x 8 tiles, a lane per tile, over segments
// of the depth order, a wave per (open group, segment): the wave reads 64
// Gaussians' rectangles at a time and hands each that covers the group to all
// lanes as a 64-bit tile mask, so a lane counts (k_extend_count) or appends
// (k_extend_write) its tile's Gaussians in depth order.  In between
// k_extend_place turns the counts into places.  With few open tiles the
// segments spread them over the chip; each open group reads every rectangle.
struct ExtendArgs {
    uint32_t prefix;
    uint64_t capacity;     // entries of point_list
    const uint32_t* n_owners;
    const uint32_t* origin;
    const uint32_t* size;
    const uint32_t* ids;
    OpenTiles open;
    uint32_t* counts;      // [groups * segments * 64]
    uint32_t* done;        // [tiles]
    int grid_x, grid_y, segments;
};

constexpr int kExtendBlocks = 1024;

// this lane's tile of group g: whether the blend left it open
__device__ __forceinline__ bool extend_lane_open(const ExtendArgs& a, int g, int* gx0, int* gy0, int* tile)
{
    const int groups_x = (a.grid_x + 7) / 8;
    *gx0 = g % groups_x * 8;
    *gy0 = g / groups_x * 8;
    const int lane = int(lane_id());
    const int tx = *gx0 + lane % 8, ty = *gy0 + lane / 8;
    *tile = ty * a.grid_x + tx;
    return tx < a.grid_x && ty < a.grid_y && ((a.open.tiles[ty * a.open.row_words + tx / 32] >> (tx % 32)) & 1u) != 0;
}

// calls f(id position, this lane's tile is covered) for the positions of segment
// `seg` that cover an open tile of the group, in order
template <class F>
__device__ __forceinline__ void extend_walk(const ExtendArgs& a, int gx0, int gy0, int seg, uint64_t open_tiles, F&& f)
{
    const uint32_t n = *a.n_owners;
    const uint32_t per = (n + uint32_t(a.segments) * 64 - 1) / (uint32_t(a.segments) * 64) * 64;
    const uint64_t k0 = uint64_t(seg) * per;
    const uint32_t k1 = uint32_t(min(uint64_t(n), k0 + per));
    const unsigned lane = lane_id();
    constexpr int U = 4; // rectangles in flight per lane
    for (uint64_t kb = k0; kb < k1; kb += 64 * U) {
        uint32_t o[U], sz[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = uint32_t(min(kb + uint64_t(64 * u) + lane, uint64_t(k1 - 1)));
            o[u] = a.origin[k];
            sz[u] = a.size[k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t kbu = kb + uint64_t(64 * u);
            uint64_t m = 0;
            if (kbu + lane < k1) {
                const int x0 = int(o[u] & 0xffffu) - gx0, y0 = int(o[u] >> 16) - gy0;
                const int x1 = min(x0 + int(sz[u] & 0xffffu), 8), y1 = min(y0 + int(sz[u] >> 16), 8);
                const int xa = max(x0, 0), ya = max(y0, 0);
                if (xa < x1 && ya < y1) {
                    const uint64_t cols = ((0xffu << xa) & (0xffu >> (8 - x1))) * 0x0101010101010101ull;
                    const uint64_t rows = (~uint64_t(0) << (8 * ya)) & (~uint64_t(0) >> (64 - 8 * y1));
                    m = cols & rows & open_tiles;
                }
            }
            for (uint64_t hit = __builtin_amdgcn_ballot_w64(m != 0); hit != 0; hit &= hit - 1) {
                const int j = __builtin_ctzll(hit);
                const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(m), j), hi = __builtin_amdgcn_readlane(uint32_t(m >> 32), j);
                f(uint32_t(kbu) + uint32_t(j), (((lane & 32u) ? hi : lo) >> (lane & 31u)) & 1u);
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_extend_count(ExtendArgs a)
{
    if (*a.open.any == 0)
        return;
    const uint32_t items = a.open.groups[0] * uint32_t(a.segments);
    for (uint32_t i = uniform(blockIdx.x * 4 + threadIdx.x / 64); i < items; i += kExtendBlocks * 4) {
        const int at = int(i / uint32_t(a.segments)), seg = int(i % uint32_t(a.segments));
        int gx0, gy0, tile;
        const bool open = extend_lane_open(a, int(a.open.groups[1 + at]), &gx0, &gy0, &tile);
        uint32_t count = 0;
        extend_walk(a, gx0, gy0, seg, __builtin_amdgcn_ballot_w64(open), [&](uint32_t, uint32_t covered) { count += covered; });
        a.counts[int64_t(i) * 64 + lane_id()] = count;
    }
}

// per open group: every (segment, tile) run's place in point_list, and the
// tiles' ranges.  A wave takes a sixteenth of the segments.
constexpr int kPlaceWaves = 16;
__global__ __launch_bounds__(64 * kPlaceWaves) void k_extend_place(ExtendArgs a, uint32_t* __restrict__ ranges)
{
    __shared__ uint32_t s_run[kPlaceWaves][64];
    __shared__ uint32_t s_fits;
    if (*a.open.any == 0)
        return;
    const unsigned lane = lane_id();
    const int wave = int(uniform(threadIdx.x / 64));
    const int per = (a.segments + kPlaceWaves - 1) / kPlaceWaves;
    const int s0 = min(a.segments, wave * per), s1 = min(a.segments, s0 + per);
    for (uint32_t at = blockIdx.x; at < a.open.groups[0]; at += gridDim.x) {
        uint32_t* rows = a.counts + int64_t(at) * a.segments * 64 + lane;
        uint32_t sum = 0;
#pragma unroll 8
        for (int s = s0; s < s1; ++s)
            sum += rows[s * 64];
        s_run[wave][lane] = sum;
        __syncthreads();
        if (wave == 0) {
            int gx0, gy0, tile;
            const bool open = extend_lane_open(a, int(a.open.groups[1 + at]), &gx0, &gy0, &tile);
            uint32_t total = 0;
            for (int w = 0; w < kPlaceWaves; ++w)
                total += s_run[w][lane];
            uint32_t before = total; // inclusive sum over the lanes
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(before, d);
                before += lane >= unsigned(d) ? v : 0u;
            }
            const uint32_t all = __shfl(before, 63);
            uint32_t base = 0;
            if (lane == 0)
                base = atomicAdd(a.open.rest, all);
            base = a.prefix + __shfl(base, 0);
            const bool fits = uint64_t(base) + all <= a.capacity; // always, unless the pairs exceed the caller's capacity
            uint32_t run = base + (before - total);
            if (open) {
                a.done[tile] = ranges[2 * tile + 1] - ranges[2 * tile];
                ranges[2 * tile] = fits && total ? run : 0u;
                ranges[2 * tile + 1] = fits && total ? run + total : 0u;
            }
            for (int w = 0; w < kPlaceWaves; ++w) {
                const uint32_t c = s_run[w][lane];
                s_run[w][lane] = run;
                run += c;
            }
            if (lane == 0)
                s_fits = fits;
        }
        __syncthreads();
        uint32_t run = s_run[wave][lane];
        const bool fits = s_fits != 0;
        for (int s = s0; s < s1; s += 8) {
            uint32_t c[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                c[u] = s + u < s1 ? rows[(s + u) * 64] : 0u;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (s + u < s1)
                    rows[(s + u) * 64] = fits ? run : 0xffffffffu;
                run += c[u];
            }
        }
        __syncthreads(); // s_run and s_fits are written again
    }
}

__global__ __launch_bounds__(256) void k_extend_write(ExtendArgs a, uint32_t* __restrict__ point_list)
{
    if (*a.open.any == 0)
        return;
    const uint32_t items = a.open.groups[0] * uint32_t(a.segments);
    for (uint32_t i = uniform(blockIdx.x * 4 + threadIdx.x / 64); i < items; i += kExtendBlocks * 4) {
        const int at = int(i / uint32_t(a.segments)), seg = int(i % uint32_t(a.segments));
        int gx0, gy0, tile;
        const bool open = extend_lane_open(a, int(a.open.groups[1 + at]), &gx0, &gy0, &tile);
        uint32_t place = a.counts[int64_t(i) * 64 + lane_id()];
        if (uniform(place) == 0xffffffffu)
            continue; // did not fit (the whole group)
        extend_walk(a, gx0, gy0, seg, __builtin_amdgcn_ballot_w64(open), [&](uint32_t k, uint32_t covered) {
            const uint32_t id = a.ids[k];
            if (covered)
                point_list[place++] = id;
        });
    }
}

template <int TW, int TH, int B, int SPLIT>
__global__ __launch_bounds__(64 * kBlendWaves) void k_blend_backward(const uint32_t* __restrict__ ranges, const uint32_t* __restrict__ point_list,
    const float2* __restrict__ xy, const float4* __restrict__ conic_opacity, const float* __restrict__ rgb, int width, int height, int grid_x,
    int n_tiles, float bg0, float bg1, float bg2, const float* __restrict__ framebuffer, const float* __restrict__ final_T,
    const float* __restrict__ grad_fb, float* __restrict__ screen_grads, WavePriority prio)
{
    __shared__ BlendSmemBwd<B> sm_all[kBlendWaves];
    const int wave = int(uniform(threadIdx.x / 64));
    const int unit = xcd_tile(blockIdx.x, gridDim.x) * kBlendWaves + wave;
    const int tile = unit / SPLIT, part = unit % SPLIT;
    if (tile >= n_tiles)
        return;
    BlendSmemBwd<B>& sm = sm_all[wave];
    const uint32_t first = uniform(ranges[2 * tile]), last = uniform(ranges[2 * tile + 1]);
    set_wave_priority(last - first, prio);
    blend_tile_backward<TW, TH / SPLIT, B>(sm, first, last, (tile % grid_x) * TW, (tile / grid_x) * TH + part * (TH / SPLIT), width, height,
        bg0, bg1, bg2, point_list, xy, conic_opacity, rgb, framebuffer, final_T, grad_fb, screen_grads);
}

namespace {

// SH gradient rows (3 * sh_coeffs floats per Gaussian, 192 B at degree 3)
// are written by the whole wave: each lane stages its Gaussian's factors
// (16 basis values, 3 colour gradients) in LDS, then the wave writes its 64
// rows as one contiguous span, 256 B per store instruction.  Per-lane row
// stores would leave lines partly written while 64 rows of every resident
// wave compete for L2, and each partial eviction is a separate HBM write.
constexpr int kShStage = 19; // odd row stride: the 64 lanes' rows hit distinct banks

__global__ __launch_bounds__(kPreThreads) void k_splat_preprocess_backward(int64_t n, SplatParams p, DevCamera<float> cam,
    const uint32_t* __restrict__ tiles, const float4* __restrict__ conic_opacity, const uint8_t* __restrict__ clamped,
    const float* __restrict__ screen_grads, float* __restrict__ g_means, float* __restrict__ g_scales, float* __restrict__ g_rotations,
    float* __restrict__ g_opacity, float* __restrict__ g_sh)
{
    __shared__ float s_stage[kPreThreads * kShStage];
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int lane = int(threadIdx.x & 63);
    const int kc = 3 * p.sh_coeffs;
    float* row = s_stage + threadIdx.x * kShStage;
    if (i < n) {
        float g_mu[3] = { 0.f, 0.f, 0.f }, g_s[3] = { 0.f, 0.f, 0.f }, g_q[4] = { 0.f, 0.f, 0.f, 0.f }, g_w = 0.f;
        if (tiles[i] != 0) {
            preprocess_backward_gaussian<ShGrad::Export>(i, p, p.sh + i * kc, cam, conic_opacity[i], clamped + 3 * i, screen_grads + i * 9,
                g_mu, g_s, g_q, &g_w, row);
        } else {
            for (int k = 0; k < kShStage; ++k)
                row[k] = 0.f;
        }
        activation_backward(p, i, g_s, g_q, &g_w);
        for (int a = 0; a < 3; ++a) {
            g_means[3 * i + a] = g_mu[a];
            g_scales[3 * i + a] = g_s[a];
        }
        for (int a = 0; a < 4; ++a)
            g_rotations[4 * i + a] = g_q[a];
        g_opacity[i] = g_w;
    }
    wave_lds_sync();
    const int64_t first = i - lane; // the wave's first Gaussian
    if (first >= n)
        return;
    const int count = int(min<int64_t>(64, n - first)) * kc;
    const float* rows = s_stage + (threadIdx.x - lane) * kShStage;
    float* dst = g_sh + first * kc;
    // f = g * kc + 3 * k + ch; the quotients come from float products, exact
    // here since f < 64 * 48 keeps every quotient 1/(2 kc) away from an integer
    const float inv_kc = 1.f / float(kc);
    for (int f = lane; f < count; f += 64) {
        const int g = int((float(f) + 0.5f) * inv_kc);
        const int e = f - g * kc;
        const int k = int((float(e) + 0.5f) * (1.f / 3.f));
        const float* r = rows + g * kShStage;
        dst[f] = r[k] * r[16 + (e - 3 * k)];
    }
}

SplatParams make_params(const dgmr_gaussians* g)
{
    return SplatParams { static_cast<const float*>(g->means), static_cast<const float*>(g->scales), static_cast<const float*>(g->rotations),
        static_cast<const float*>(g->opacity), static_cast<const float*>(g->sh), g->sh_coeffs, g->sh_degree, float(g->scale_multiplier),
        g->activation };
}

} // namespace

SplatParams make_splat_params(const dgmr_gaussians* g) { return make_params(g); }

hipError_t launch_splat_preprocess(const dgmr_gaussians* g, const DevCamera<float>& cam, const SplatOut& out, hipStream_t stream)
{
    k_splat_preprocess<<<unsigned(ceil_div64(g->n, kPreThreads)), kPreThreads, 0, stream>>>(g->n, make_params(g), cam, out);
    return hipGetLastError();
}

namespace {
// one wave: out[l] = wave_sum8 of in[q * 64 + l] (q < 8), out[64 + l] = wave_sum_to_last of in[512 + l]
__global__ __launch_bounds__(64) void k_selftest_wave_sum(const float* __restrict__ in, float* __restrict__ out)
{
    const int l = int(threadIdx.x);
    out[l] = wave_sum8(in[l], in[64 + l], in[128 + l], in[192 + l], in[256 + l], in[320 + l], in[384 + l], in[448 + l]);
    out[64 + l] = wave_sum_to_last(in[512 + l]);
}

} // namespace

// ------------------------------------------------------------------ host side
struct SplatWorkspace {
    uint32_t* dkeys_a;
    uint32_t* dvals_a;
    uint32_t* dkeys_b;
    uint32_t* dvals_b;
    uint32_t* counts;
    uint32_t* emit_bounds;
    uint2* owner_rects;   // without tight culling
    uint2* bin_rects;
    ReachRec* owner_reach; // with tight culling (the same memory as owner_rects / bin_rects)
    ReachRec* reach;
    uint32_t* pair_offsets;
    uint32_t* pkeys_a;
    uint32_t* pvals_a;
    uint32_t* pkeys_b;
    uint32_t* counter;
    void* sort_scratch;
    void* scan_scratch;
};

static SplatWorkspace carve_splat(Carver& cv, int64_t n, int64_t cap, bool cull)
{
    SplatWorkspace w;
    const int64_t nn = std::max<int64_t>(n, 1), cc = std::max<int64_t>(cap, 1);
    const int64_t rec = cull ? int64_t(sizeof(ReachRec)) : int64_t(sizeof(uint2)); // bytes per Gaussian record
    w.dkeys_a = cv.take<uint32_t>(nn);
    w.dvals_a = cv.take<uint32_t>(nn);
    w.reach = reinterpret_cast<ReachRec*>(cv.take<char>(nn * rec));
    w.bin_rects = reinterpret_cast<uint2*>(w.reach);
    w.dkeys_b = cv.take<uint32_t>(nn);
    w.dvals_b = cv.take<uint32_t>(nn);
    w.counts = cv.take<uint32_t>(nn);
    w.pair_offsets = cv.take<uint32_t>(nn);
    w.pkeys_a = cv.take<uint32_t>(cc);
    w.pvals_a = cv.take<uint32_t>(cc);
    w.pkeys_b = cv.take<uint32_t>(cc);
    w.counter = cv.take<uint32_t>(64);
    w.emit_bounds = cv.take<uint32_t>(cc / (kEmitThreads * kEmitPerSmall) + 2);
    w.owner_reach = reinterpret_cast<ReachRec*>(cv.take<char>(nn * rec));
    w.owner_rects = reinterpret_cast<uint2*>(w.owner_reach);
    w.sort_scratch = cv.take<char>(radix_scratch_bytes(std::max(nn, cc)));
    w.scan_scratch = cv.take<char>(scan_scratch_bytes(nn, 2));
    return w;
}

size_t splat_workspace_bytes(int64_t n, int64_t cap, bool cull)
{
    Carver cv(nullptr, 0);
    carve_splat(cv, n, cap, cull);
    return cv.used;
}

template <int TW, int TH, int SPLIT>
static void launch_blend_fwd_as(int batch, int n_tiles, hipStream_t st, const uint32_t* ranges, const uint32_t* pl, const float2* xy,
    const float4* co, const float* rgb, int W, int H, int gx, const double* bg, float* fb, float* T, const PrefixPass& prefix)
{
    const dim3 grid(unsigned(ceil_div64(int64_t(n_tiles) * SPLIT, kBlendWaves))), block(64 * kBlendWaves);
    const float b0 = float(bg[0]), b1 = float(bg[1]), b2 = float(bg[2]);
    if (batch == 64)
        k_blend_forward<TW, TH, 64, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, prefix);
    else if (batch == 128)
        k_blend_forward<TW, TH, 128, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, prefix);
    else
        k_blend_forward<TW, TH, 256, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, prefix);
}

template <int TW, int TH>
static void launch_blend_fwd(int batch, int n_tiles, hipStream_t st, const uint32_t* ranges, const uint32_t* pl, const float2* xy,
    const float4* co, const float* rgb, int W, int H, int gx, const double* bg, float* fb, float* T, const PrefixPass& prefix)
{
    // the second pass of prefix binning mostly has few tiles to blend
    constexpr int SPLIT = TW * TH / 64;
    if (SPLIT > 1 && (n_tiles <= kFwdSplitTiles || prefix.again))
        launch_blend_fwd_as<TW, TH, SPLIT>(batch, n_tiles, st, ranges, pl, xy, co, rgb, W, H, gx, bg, fb, T, prefix);
    else
        launch_blend_fwd_as<TW, TH, 1>(batch, n_tiles, st, ranges, pl, xy, co, rgb, W, H, gx, bg, fb, T, prefix);
}

template <int TW, int TH, int SPLIT>
static void launch_blend_bwd_as(int batch, int n_tiles, hipStream_t st, const uint32_t* ranges, const uint32_t* pl, const float2* xy,
    const float4* co, const float* rgb, int W, int H, int gx, const double* bg, const float* fb, const float* T, const float* gfb, float* sg,
    WavePriority prio)
{
    const dim3 grid(unsigned(ceil_div64(int64_t(n_tiles) * SPLIT, kBlendWaves))), block(64 * kBlendWaves);
    const float b0 = float(bg[0]), b1 = float(bg[1]), b2 = float(bg[2]);
    if (batch == 64)
        k_blend_backward<TW, TH, 64, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, gfb, sg, prio);
    else if (batch == 128)
        k_blend_backward<TW, TH, 128, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, gfb, sg, prio);
    else
        k_blend_backward<TW, TH, 256, SPLIT><<<grid, block, 0, st>>>(ranges, pl, xy, co, rgb, W, H, gx, n_tiles, b0, b1, b2, fb, T, gfb, sg, prio);
}

template <int TW, int TH>
static void launch_blend_bwd(int batch, int n_tiles, hipStream_t st, const uint32_t* ranges, const uint32_t* pl, const float2* xy,
    const float4* co, const float* rgb, int W, int H, int gx, const double* bg, const float* fb, const float* T, const float* gfb, float* sg,
    WavePriority prio)
{
    constexpr int SPLIT = TW * TH / 64;
    if (SPLIT > 1 && n_tiles <= kBwdSplitTiles)
        launch_blend_bwd_as<TW, TH, SPLIT>(batch, n_tiles, st, ranges, pl, xy, co, rgb, W, H, gx, bg, fb, T, gfb, sg, prio);
    else
        launch_blend_bwd_as<TW, TH, 1>(batch, n_tiles, st, ranges, pl, xy, co, rgb, W, H, gx, bg, fb, T, gfb, sg, prio);
}

// waves per tile of the forward blend (of prefix binning's first pass)
static int blend_forward_split(const dgmr_tiling& t, int64_t n_tiles) { return n_tiles <= kFwdSplitTiles ? t.tile_w * t.tile_h / 64 : 1; }

void splat_blend_forward(const dgmr_tiling& t, int n_tiles, hipStream_t st, const uint32_t* ranges, const uint32_t* pl, const float* xy,
    const float* co, const float* rgb, int W, int H, int gx, const double* bg, float* fb, float* T, const PrefixPass& prefix = PrefixPass {})
{
    const auto* xy2 = reinterpret_cast<const float2*>(xy);
    const auto* co4 = reinterpret_cast<const float4*>(co);
    if (t.tile_w == 16)
        launch_blend_fwd<16, 16>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, prefix);
    else if (t.tile_w == 8)
        launch_blend_fwd<8, 8>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, prefix);
    else
        launch_blend_fwd<32, 8>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, prefix);
}

void splat_blend_backward(const dgmr_tiling& t, int n_tiles, int64_t n_pairs, hipStream_t st, const uint32_t* ranges, const uint32_t* pl,
    const float* xy, const float* co, const float* rgb, int W, int H, int gx, const double* bg, const float* fb, const float* T, const float* gfb,
    float* sg)
{
    const auto* xy2 = reinterpret_cast<const float2*>(xy);
    const auto* co4 = reinterpret_cast<const float4*>(co);
    // priority thresholds at 0.55, 0.93 and 1.37 times the mean list length
    // (1M Gaussians at 1080p: blend backward 0.210 -> 0.200 ms)
    const double mean = double(n_pairs) / double(std::max(n_tiles, 1));
    const auto at = [&](double f) { return uint32_t(std::min(f * mean, double(UINT32_MAX))); };
    const WavePriority prio { at(0.55), at(0.93), at(1.37) };
    if (t.tile_w == 16)
        launch_blend_bwd<16, 16>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, gfb, sg, prio);
    else if (t.tile_w == 8)
        launch_blend_bwd<8, 8>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, gfb, sg, prio);
    else
        launch_blend_bwd<32, 8>(t.batch, n_tiles, st, ranges, pl, xy2, co4, rgb, W, H, gx, bg, fb, T, gfb, sg, prio);
}

static OpenTiles open_tiles(const PrefixBinning& p) { return OpenTiles { p.open_tiles, p.row_words, p.open_words, p.any_open, p.positions, p.rest, p.groups, p.group_noted }; }

struct EmitArgs {
    int64_t n;
    unsigned blocks_n;
    uint32_t cap;
    int64_t n_tiles;
    int tile_bits;
    const uint32_t* sorted_ids;
    const int4* views;
    int64_t n_per_view;
    int n_views;
    int tile_w, tile_h;
    bool cull;
    const PrefixBinning* prefix; // null: whole lists
    bool bounds_written;         // by the small views' binning
};

// pairs: the most that are emitted, with prefix binning in its first round
static int emit_per(int64_t pairs) { return pairs >= kEmitLarge ? kEmitPerLarge : kEmitPerSmall; }
static int emit_shift(int per) { return __builtin_ctz(unsigned(kEmitThreads * per)); } // log2 of a block's pairs

// the buffer pairs of emission and pair sort, so that the sorted ids end in `list`
template <class KeyT>
static SortBuffersT<KeyT> pair_buffers(const SplatWorkspace& w, uint32_t* list, int passes)
{
    KeyT* ka = reinterpret_cast<KeyT*>(w.pkeys_a);
    KeyT* kb = reinterpret_cast<KeyT*>(w.pkeys_b);
    return passes % 2 == 0 ? SortBuffersT<KeyT> { ka, list, kb, w.pvals_a } : SortBuffersT<KeyT> { ka, w.pvals_a, kb, list };
}

// emission of *n_emit pairs
template <class KeyT>
static int launch_emit(const EmitArgs& a, const SplatWorkspace& w, const uint32_t* n_emit, const uint32_t* offsets, int per,
    const SortBuffersT<KeyT>& pb, hipStream_t st)
{
    const unsigned emit_blocks = unsigned(ceil_div64(a.cap, kEmitThreads * per));
    if (a.cull && per == kEmitPerLarge)
        k_emit_reach<KeyT, kEmitPerLarge><<<emit_blocks, kEmitThreads, 0, st>>>(n_emit, a.cap, a.sorted_ids, w.emit_bounds,
            offsets, w.owner_reach, a.tile_w, a.tile_h, pb.keys_a, pb.vals_a);
    else if (a.cull)
        k_emit_reach<KeyT, kEmitPerSmall><<<emit_blocks, kEmitThreads, 0, st>>>(n_emit, a.cap, a.sorted_ids, w.emit_bounds,
            offsets, w.owner_reach, a.tile_w, a.tile_h, pb.keys_a, pb.vals_a);
    else if (per == kEmitPerLarge)
        k_emit_pairs<KeyT, kEmitPerLarge><<<emit_blocks, kEmitThreads, 0, st>>>(a.n, n_emit, a.cap, a.sorted_ids, w.emit_bounds,
            offsets, w.owner_rects, pb.keys_a, pb.vals_a);
    else
        k_emit_pairs<KeyT, kEmitPerSmall><<<emit_blocks, kEmitThreads, 0, st>>>(a.n, n_emit, a.cap, a.sorted_ids, w.emit_bounds,
            offsets, w.owner_rects, pb.keys_a, pb.vals_a);
    DGMR_HIP_CHECK(hipGetLastError());
    return DGMR_OK;
}

// emission, pair sort on the tile bits, tile ranges; pair keys of type KeyT
template <class KeyT>
static int emit_sort_ranges(const EmitArgs& a, const SplatWorkspace& w, dgmr_binning* bins, PendingCount* pending, hipStream_t st)
{
    const int passes = radix_passes(0, a.tile_bits);
    const SortBuffersT<KeyT> pb = pair_buffers<KeyT>(w, bins->point_list, passes);
    const uint32_t* n_emit = a.prefix ? a.prefix->n_emit : w.counter;
    // fewer than kPrefixMin times the prefix are emitted whole
    const int per = emit_per(a.prefix ? std::min<int64_t>(a.cap, kPrefixMin * a.prefix->pairs) : a.cap);
    {
        StageScope sc("bin.emit", st);
        pending->add_stage(sc.slot, 4.0 + sizeof(KeyT), 28.0 * double(a.n));
        if (!a.bounds_written)
            k_emit_bounds<<<a.blocks_n, 256, 0, st>>>(a.n, w.pair_offsets, w.counter, a.cap, n_emit, emit_shift(per), w.emit_bounds);
        DGMR_HIP_CHECK(hipGetLastError());
        const int rc = launch_emit<KeyT>(a, w, n_emit, w.pair_offsets, per, pb, st);
        if (rc != DGMR_OK)
            return rc;
    }
    {
        StageScope sc("bin.pair_sort", st);
        pending->add_stage(sc.slot, (8.0 + 3.0 * sizeof(KeyT)) * passes, 0.0);
        DGMR_HIP_CHECK(radix_sort_pairs(pb, a.cap, n_emit, 0, a.tile_bits, w.sort_scratch, st));
    }
    const KeyT* sorted_keys = (passes % 2 == 0) ? pb.keys_a : pb.keys_b;
    const uint32_t* sorted_vals = (passes % 2 == 0) ? pb.vals_a : pb.vals_b;
    {
        StageScope sc("bin.ranges", st);
        pending->add_stage(sc.slot, 0.0, 8.0 * double(a.n_tiles));
        k_tile_ranges<KeyT><<<unsigned(ceil_div64(a.n_tiles, 256)), 256, 0, st>>>(sorted_keys, sorted_vals, n_emit, a.cap, a.views,
            a.n_views, a.n_per_view, a.n_tiles, bins->ranges, a.prefix ? open_tiles(*a.prefix) : OpenTiles {});
        DGMR_HIP_CHECK(hipGetLastError());
    }
    return DGMR_OK;
}

// the whole lists of the open tiles behind the prefixes (nothing when there are none)
template <class KeyT>
static int extend_lists_keyed(const EmitArgs& a, const SplatWorkspace& w, dgmr_binning* bins, hipStream_t st)
{
    const PrefixBinning& p = *a.prefix;
    const OpenTiles open = open_tiles(p);
    const unsigned blocks = unsigned(ceil_div64(a.n, 256 * kOpenPer));
    const ScanState scan = scan_state(w.scan_scratch, a.n, 2);
    if (open.words <= kOpenLdsWords)
        k_open_owners<true><<<blocks, 256, size_t(open.words) * sizeof(uint32_t), st>>>(open, p.grid_x, p.n_owners, p.origin, p.size, w.counts,
            p.flags, scan);
    else
        k_open_owners<false><<<blocks, 256, 0, st>>>(open, p.grid_x, p.n_owners, p.origin, p.size, w.counts, p.flags, scan);
    DGMR_HIP_CHECK(hipGetLastError());
    const ScanArray scans[2] = { { w.counts, w.pair_offsets, open.rest, false }, { p.flags, p.flags, nullptr, false } };
    DGMR_HIP_CHECK(scan_u32_arrays(scans, 2, a.n, w.scan_scratch, st, true, ScanLength { open.positions, 1, 1 }));
    k_open_bounds<<<blocks, 256, 0, st>>>(open, w.pair_offsets, p.flags, p.origin, p.size, p.ids, p.grid_x, a.cap, emit_shift(kEmitPerSmall),
        w.counts, w.owner_rects, p.ids_out, w.emit_bounds);
    DGMR_HIP_CHECK(hipGetLastError());
    const int passes = radix_passes(0, a.tile_bits);
    const SortBuffersT<KeyT> pb = pair_buffers<KeyT>(w, bins->point_list + p.pairs, passes);
    const int rc = launch_emit<KeyT>(a, w, open.rest, w.counts, kEmitPerSmall, pb, st);
    if (rc != DGMR_OK)
        return rc;
    DGMR_HIP_CHECK(radix_sort_pairs(pb, a.cap, open.rest, 0, a.tile_bits, w.sort_scratch, st));
    k_open_ranges<KeyT><<<unsigned(ceil_div64(a.n_tiles, 256)), 256, 0, st>>>((passes % 2 == 0) ? pb.keys_a : pb.keys_b, a.cap, p.pairs, open,
        p.grid_x, a.n_tiles, bins->ranges, p.done);
    DGMR_HIP_CHECK(hipGetLastError());
    return DGMR_OK;
}

static int extend_lists(const PrefixBinning& p, bool few, int64_t n, int64_t n_tiles, void* workspace, size_t workspace_bytes, dgmr_binning* bins,
    hipStream_t st)
{
    StageScope sc(few ? "bin.extend_few" : "bin.extend", st);
    Carver cv(workspace, workspace_bytes);
    const SplatWorkspace w = carve_splat(cv, n, bins->pair_capacity, false); // as the binning carved it
    const int64_t cap = std::min<int64_t>(bins->pair_capacity, int64_t(UINT32_MAX));
    if (few) {
        // the pair keys are not read again: their buffer holds the counts
        const int grid_y = int(n_tiles / p.grid_x);
        const int64_t groups = ceil_div64(p.grid_x, 8) * ceil_div64(grid_y, 8);
        const int segments = int(std::min<int64_t>(512, cap / (groups * 64)));
        const ExtendArgs xa { p.pairs, uint64_t(p.pairs + cap), p.n_owners, p.origin, p.size, p.ids, open_tiles(p), w.pkeys_a, p.done, p.grid_x, grid_y,
            segments };
        k_extend_count<<<kExtendBlocks, 256, 0, st>>>(xa);
        DGMR_HIP_CHECK(hipGetLastError());
        k_extend_place<<<unsigned(std::min<int64_t>(groups, 256)), 64 * kPlaceWaves, 0, st>>>(xa, bins->ranges);
        DGMR_HIP_CHECK(hipGetLastError());
        k_extend_write<<<kExtendBlocks, 256, 0, st>>>(xa, bins->point_list);
        DGMR_HIP_CHECK(hipGetLastError());
        return DGMR_OK;
    }
    const EmitArgs ea { n, unsigned(ceil_div64(n, 256)), uint32_t(cap), n_tiles, int(higher_msb(uint32_t(n_tiles))), p.ids_out, nullptr, 0, 0, 0, 0, false, &p,
        false };
    return ea.tile_bits <= 16 ? extend_lists_keyed<uint16_t>(ea, w, bins, st) : extend_lists_keyed<uint32_t>(ea, w, bins, st);
}

// binning shared by the splatter and the marcher: depth sort, scan, emission,
// pair sort, ranges.  depth_keys/ids are the workspace's A buffers, filled by
// the preprocess.  Returns the pair count through *n_pairs (host).
int bin_gaussians(int64_t n, const int32_t* rects, const uint32_t* tiles, const void* xy, bool xy_double, bool bin_rects_written, bool cull,
    int grid_x, int grid_y, int tile_w, int tile_h, dgmr_binning* bins, Carver& cv, PendingCount* pending, hipStream_t st,
    const BatchBinning* batch, PrefixBinning* prefix)
{
    const int4* views = batch ? batch->views : nullptr;
    const int64_t n_per_view = batch ? batch->n_per_view : 0;
    SplatWorkspace w = carve_splat(cv, n, bins->pair_capacity, cull);
    // stable sort of Gaussian ids by depth bits.  Large sorts first keep only
    // the visible entries (culled ones carry the key 0xffffffff and would sort
    // last anyway), in order, so the sort and everything after it sees fewer
    // keys; n_sorted (device) is then their count.
    uint32_t *K = w.dkeys_a, *V = w.dvals_a, *K2 = w.dkeys_b, *V2 = w.dvals_b;
    const uint32_t* n_sorted = nullptr;
    if (n >= kCompactMin) {
        StageScope sc("bin.compact", st, 16.0 * double(n));
        uint32_t* count = w.counter + 1;
        // the preprocess left the ids unwritten: the compaction numbers the entries
        DGMR_HIP_CHECK(compact_pairs(K, nullptr, n, 0xffffffffu, K2, V2, count, w.counts, w.pair_offsets, w.scan_scratch, st));
        std::swap(K, K2);
        std::swap(V, V2);
        n_sorted = count;
    }
    const bool multi_view = batch && batch->n_views > 1;
    const bool one = bin_rects_written && !cull && !batch && !prefix && n <= kBinOneMax;
    // with tight culling the culled entries sort last in the view pass, under the key n_views
    const uint32_t culled_view = cull && multi_view ? uint32_t(batch->n_views) : 0xffffffffu;
    if (!one) {
        StageScope sc("bin.depth_sort", st, 16.0 * double(n) * radix_passes(0, 32));
        // several views: the last depth pass writes each entry's view as its key
        const KeyOut view_keys = multi_view ? KeyOut { uint32_t(n_per_view), culled_view } : KeyOut {};
        DGMR_HIP_CHECK(radix_sort_pairs(SortBuffers { K, V, K2, V2 }, n, n_sorted, 0, 32, w.sort_scratch, st, view_keys));
        if (radix_passes(0, 32) % 2 == 1) {
            std::swap(K, K2);
            std::swap(V, V2);
        }
    }
    if (multi_view) {
        // stable pass on the view index: order becomes (view, depth bits, id)
        StageScope sc("bin.view_sort", st, 16.0 * double(n));
        const int vbits = int(higher_msb(cull ? uint32_t(batch->n_views) : uint32_t(batch->n_views - 1)));
        DGMR_HIP_CHECK(radix_sort_pairs(SortBuffers { K, V, K2, V2 }, n, n_sorted, 0, vbits, w.sort_scratch, st));
        if (radix_passes(0, vbits) % 2 == 1) {
            std::swap(K, K2);
            std::swap(V, V2);
        }
    }
    const uint32_t* sorted_ids = V;
    // prefix binning: the sorted depth keys are not read again, their buffers
    // hold the rectangles; nor, once gathered, the records in id order, whose
    // 2 n words hold what the blend notes (8 per tile and one, and n >= 96 per tile)
    // and the extension's flags
    PrefixRects rects_out { nullptr, nullptr, nullptr };
    if (prefix) {
        static_assert(kPrefixMin * kPrefixPerTile * sizeof(uint32_t) >= sizeof(DecideSums), "the pair keys' buffer holds the sums until the emission");
        rects_out = PrefixRects { K, K2, reinterpret_cast<DecideSums*>(w.pkeys_a) };
        const int64_t n_tiles = int64_t(grid_x) * grid_y;
        uint32_t* words = reinterpret_cast<uint32_t*>(w.bin_rects);
        prefix->ids = sorted_ids;
        prefix->ids_out = V2;
        prefix->origin = K;
        prefix->size = K2;
        prefix->n_pairs = w.counter;
        prefix->n_emit = w.counter + 2;
        prefix->few = w.counter + 3;
        prefix->n_owners = w.counter + 4;
        prefix->any_open = w.counter + 5;
        prefix->positions = w.counter + 6;
        prefix->rest = w.counter + 7;
        prefix->units = words;
        prefix->done = words + 4 * n_tiles;
        prefix->open_tiles = words + 5 * n_tiles;
        prefix->group_noted = words + 6 * n_tiles;
        prefix->groups = words + 7 * n_tiles;
        prefix->flags = words + (8 * n_tiles + 1 + 3) / 4 * 4;
        prefix->grid_x = grid_x;
        prefix->row_words = int(ceil_div64(grid_x, 32));
        prefix->open_words = int64_t(prefix->row_words) * grid_y;
    }
    const unsigned blocks_n = unsigned(ceil_div64(n, 256));
    const int64_t cap = std::min<int64_t>(bins->pair_capacity, int64_t(UINT32_MAX));
    if (one) {
        StageScope sc("bin.one", st, 60.0 * double(n));
        k_bin_one<<<bins->point_offsets ? 2 : 1, kBinOneThreads, 0, st>>>(BinOneArgs { int(n), K, w.bin_rects, tiles, uint32_t(grid_x), uint32_t(std::max<int64_t>(cap, 0)),
            emit_shift(emit_per(cap)), V, w.owner_rects, w.pair_offsets, bins->point_offsets, w.counter, w.emit_bounds });
        DGMR_HIP_CHECK(hipGetLastError());
    } else {
        StageScope sc("bin.scan", st, 44.0 * double(n));
        // the pair offsets of the depth order and, when asked for, the
        // reference cache's inclusive scan of tiles in Gaussian order: one
        // launch, its state cleared by the gather (one thread per item)
        const ScanArray scans[2] = { { w.counts, w.pair_offsets, w.counter, false }, { tiles, bins->point_offsets, nullptr, true } };
        const int n_scans = bins->point_offsets ? 2 : 1;
        const ScanState scan = scan_state(w.scan_scratch, n, n_scans);
        if (cull)
            k_gather_reach<<<blocks_n, 256, 0, st>>>(n, n_sorted, K, batch && batch->n_views > 1 ? uint32_t(batch->n_views) : 0xffffffffu,
                sorted_ids, w.reach, tile_w, tile_h, w.counts, w.owner_reach, scan);
        else if (bin_rects_written)
            k_gather_owners<float, true><<<blocks_n, 256, 0, st>>>(n, n_sorted, sorted_ids, w.bin_rects, rects, tiles, static_cast<const float*>(xy),
                grid_x, grid_y, tile_w, tile_h, views, n_per_view, w.counts, w.owner_rects, scan, rects_out);
        else if (xy_double)
            k_gather_owners<double, false><<<blocks_n, 256, 0, st>>>(n, n_sorted, sorted_ids, w.bin_rects, rects, tiles,
                static_cast<const double*>(xy), grid_x, grid_y, tile_w, tile_h, views, n_per_view, w.counts, w.owner_rects, scan, rects_out);
        else
            k_gather_owners<float, false><<<blocks_n, 256, 0, st>>>(n, n_sorted, sorted_ids, w.bin_rects, rects, tiles,
                static_cast<const float*>(xy), grid_x, grid_y, tile_w, tile_h, views, n_per_view, w.counts, w.owner_rects, scan, rects_out);
        DGMR_HIP_CHECK(hipGetLastError());
        DGMR_HIP_CHECK(scan_u32_arrays(scans, n_scans, n, w.scan_scratch, st, true));
    }
    // R stays on the device: the copy to the host is awaited by the caller
    if (prefix) {
        k_prefix_decide<<<kDecideBlocks, kDecideThreads, 0, st>>>(DecideArgs { n, w.pair_offsets, w.counter, uint32_t(cap), prefix->pairs, prefix->always,
            sorted_ids, prefix->origin, prefix->size, prefix->conic_opacity, grid_x, grid_y, tile_w * tile_h, rects_out.sums, prefix->n_emit, prefix->few, prefix->n_owners });
        DGMR_HIP_CHECK(hipGetLastError());
    }
    const int rc_count = enqueue_count(w.counter, st, pending, prefix ? int(prefix->n_emit - w.counter) : 0);
    if (rc_count != DGMR_OK)
        return rc_count;
    const int64_t n_tiles = batch ? batch->total_tiles : int64_t(grid_x) * grid_y;
    if (cap <= 0) {
        DGMR_HIP_CHECK(hipMemsetAsync(bins->ranges, 0, size_t(n_tiles) * 2 * sizeof(uint32_t), st));
        return DGMR_OK;
    }
    // view-local tile ids as keys: 16 bits when they fit (a quarter less
    // traffic in emission and sort), else 32
    const int tile_bits = int(higher_msb(uint32_t(batch ? batch->max_view_tiles : n_tiles)));
    EmitArgs ea { n, blocks_n, uint32_t(cap), n_tiles, tile_bits, sorted_ids, views, n_per_view, batch ? int(batch->n_views) : 0, tile_w, tile_h,
        cull, prefix, one };
    if (tile_bits <= 16)
        return emit_sort_ranges<uint16_t>(ea, w, bins, pending, st);
    return emit_sort_ranges<uint32_t>(ea, w, bins, pending, st);
}

// depth keys / ids buffers the preprocess writes and its per-Gaussian
// binning records (the first three slices of carve_splat)
void binning_key_buffers(void* workspace, int64_t n, bool cull, uint32_t** keys, uint32_t** ids, void** records)
{
    // these slices come first, so they do not depend on the pair capacity
    Carver cv(workspace, ~size_t(0));
    const SplatWorkspace w = carve_splat(cv, n, 1, cull);
    *keys = w.dkeys_a;
    // sorts that compact first take the entry index as the id
    *ids = n >= kCompactMin ? nullptr : w.dvals_a;
    if (records)
        *records = w.reach;
}

} // namespace dgmr

using namespace dgmr;

static int splat_forward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, dgmr_splat_geometry* geom,
    dgmr_binning* bins, float* framebuffer, float* final_transmittance, void* workspace, size_t workspace_bytes, dgmr_stats* stats,
    dgmr_stream stream, int32_t lists, int64_t* n_binned)
{
    DGMR_ARG_CHECK(g && cam && geom && bins && framebuffer && final_transmittance && workspace, "dgmr_splat_forward: null argument");
    DGMR_ARG_CHECK(g->dtype == DGMR_F32, "dgmr_splat_forward: the splatter computes in float32");
    DGMR_ARG_CHECK(valid_tiling(tiling), "dgmr_splat_forward: tiling must be 8x8, 16x16 or 32x8 with batch 64/128/256");
    DGMR_ARG_CHECK(g->n >= 0 && g->n < (int64_t(1) << 31), "dgmr_splat_forward: bad Gaussian count");
    DGMR_ARG_CHECK(g->sh_coeffs >= 1 && g->sh_coeffs <= 16 && g->sh_degree >= 0 && g->sh_degree <= 3, "dgmr_splat_forward: bad SH layout");
    DGMR_ARG_CHECK(valid_image(cam->width, cam->height), "dgmr_splat_forward: bad image size");
    DGMR_ARG_CHECK(bins->point_list && bins->ranges, "dgmr_splat_forward: null binning buffers");
    const int64_t n = g->n;
    const bool cull = tiling->cull != 0;
    DGMR_ARG_CHECK(workspace_bytes >= splat_workspace_bytes(n, bins->pair_capacity, cull), "dgmr_splat_forward: workspace too small");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const DevCamera<float> dc = make_dev_camera<float>(*cam, *tiling);
    const int64_t n_tiles = int64_t(dc.grid_x) * dc.grid_y;
    const int64_t plane = int64_t(cam->width) * cam->height;
    if (stats) {
        stats->n_pairs = 0;
        stats->n_visible = 0;
    }
    if (n_binned)
        *n_binned = 0;
    if (n == 0) {
        DGMR_HIP_CHECK(hipMemsetAsync(bins->ranges, 0, size_t(n_tiles) * 2 * sizeof(uint32_t), st));
        splat_blend_forward(*tiling, int(n_tiles), st, bins->ranges, bins->point_list, geom->xy, geom->conic_opacity, geom->rgb, cam->width,
            cam->height, dc.grid_x, cam->background, framebuffer, final_transmittance);
        DGMR_HIP_CHECK(hipGetLastError());
        return DGMR_OK;
    }
    uint32_t *dkeys, *dids;
    void* recs;
    binning_key_buffers(workspace, n, cull, &dkeys, &dids, &recs);
    {
    StageScope sc("splat.preprocess", st, double(n) * (44.0 + 12.0 * g->sh_coeffs + 75.0));
    k_splat_preprocess<<<unsigned(ceil_div64(n, kPreThreads)), kPreThreads, 0, st>>>(n, make_params(g), dc,
        SplatOut { geom->rects, geom->tiles_touched, geom->xy, reinterpret_cast<float4*>(geom->conic_opacity), geom->rgb, geom->rgb_clamped,
            geom->depths, dkeys, dids, cull ? nullptr : static_cast<uint2*>(recs), cull ? static_cast<ReachRec*>(recs) : nullptr });
    DGMR_HIP_CHECK(hipGetLastError());
    }
    Carver cv(workspace, workspace_bytes);
    PendingCount pending;
    PrefixBinning pb {};
    pb.always = lists == DGMR_LISTS_PREFIX;
    pb.conic_opacity = reinterpret_cast<const float4*>(geom->conic_opacity);
    pb.pairs = lists != DGMR_LISTS_WHOLE && !cull ? uint32_t(prefix_pairs(n, n_tiles, bins->pair_capacity)) : 0u;
    const bool prefix = pb.pairs != 0;
    const int rc = bin_gaussians(n, geom->rects, geom->tiles_touched, geom->xy, false, true, cull, dc.grid_x, dc.grid_y, dc.tile_w, dc.tile_h, bins,
        cv, &pending, st, nullptr, prefix ? &pb : nullptr);
    if (rc != DGMR_OK)
        return rc;
    int blend_slot = -1;
    PrefixPass pass { pb.units, open_tiles(pb), pb.done, pb.n_pairs, pb.n_emit, pb.pairs, blend_forward_split(*tiling, n_tiles), false };
    {
        StageScope sc("splat.blend_forward", st);
        blend_slot = sc.slot;
        splat_blend_forward(*tiling, int(n_tiles), st, bins->ranges, bins->point_list, geom->xy, geom->conic_opacity, geom->rgb, cam->width,
            cam->height, dc.grid_x, cam->background, framebuffer, final_transmittance, pass);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    pending.add_stage(blend_slot, 40.0, 16.0 * double(plane) + 8.0 * double(n_tiles));
    // every launch is queued: now wait for the pair count (the extension, which
    // needs it, follows while the emission, sort and blend still run)
    const int64_t R = pending.wait();
    if (R < 0)
        return DGMR_ERR_DEVICE;
    if (stats)
        stats->n_pairs = R;
    if (n_binned)
        *n_binned = pending.binned;
    if (R > bins->pair_capacity) {
        set_error("pair capacity too small");
        return DGMR_ERR_CAPACITY;
    }
    if (prefix && pending.binned < R) {
        const int rc_ext = extend_lists(pb, pending.few, n, n_tiles, workspace, workspace_bytes, bins, st);
        if (rc_ext != DGMR_OK)
            return rc_ext;
        StageScope sc("splat.blend_open", st);
        pass.again = true;
        splat_blend_forward(*tiling, int(n_tiles), st, bins->ranges, bins->point_list, geom->xy, geom->conic_opacity, geom->rgb, cam->width,
            cam->height, dc.grid_x, cam->background, framebuffer, final_transmittance, pass);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    return DGMR_OK;
}

extern "C" {

int dgmr_workspace_size(int64_t n, int32_t width, int32_t height, const dgmr_tiling* tiling, int64_t pair_capacity, size_t* bytes)
{
    DGMR_ARG_CHECK(bytes && n >= 0 && valid_image(width, height) && valid_tiling(tiling) && pair_capacity >= 0, "dgmr_workspace_size: bad argument");
    *bytes = splat_workspace_bytes(n, pair_capacity, tiling->cull != 0);
    return DGMR_OK;
}

int dgmr_splat_forward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, dgmr_splat_geometry* geom,
    dgmr_binning* bins, float* framebuffer, float* final_transmittance, void* workspace, size_t workspace_bytes, dgmr_stats* stats,
    dgmr_stream stream)
{
    return splat_forward(g, cam, tiling, geom, bins, framebuffer, final_transmittance, workspace, workspace_bytes, stats, stream,
        DGMR_LISTS_WHOLE, nullptr);
}

int dgmr_splat_prefix_pairs(int64_t n, int32_t width, int32_t height, const dgmr_tiling* tiling, int64_t pair_capacity, int64_t* pairs)
{
    DGMR_ARG_CHECK(pairs && n >= 0 && n < (int64_t(1) << 31) && valid_image(width, height) && valid_tiling(tiling) && pair_capacity >= 0,
        "dgmr_splat_prefix_pairs: bad argument");
    const int64_t n_tiles = ceil_div64(width, tiling->tile_w) * ceil_div64(height, tiling->tile_h);
    *pairs = tiling->cull ? 0 : prefix_pairs(n, n_tiles, pair_capacity);
    return DGMR_OK;
}

int dgmr_splat_forward_prefix(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, dgmr_splat_geometry* geom,
    dgmr_binning* bins, float* framebuffer, float* final_transmittance, void* workspace, size_t workspace_bytes, dgmr_stats* stats,
    dgmr_stream stream)
{
    return splat_forward(g, cam, tiling, geom, bins, framebuffer, final_transmittance, workspace, workspace_bytes, stats, stream,
        DGMR_LISTS_PREFIX, nullptr);
}

int dgmr_splat_forward_lists(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, dgmr_splat_geometry* geom,
    dgmr_binning* bins, float* framebuffer, float* final_transmittance, void* workspace, size_t workspace_bytes, int32_t lists, int64_t* n_binned,
    dgmr_stats* stats, dgmr_stream stream)
{
    DGMR_ARG_CHECK(lists >= DGMR_LISTS_WHOLE && lists <= DGMR_LISTS_AUTO, "dgmr_splat_forward_lists: bad lists");
    return splat_forward(g, cam, tiling, geom, bins, framebuffer, final_transmittance, workspace, workspace_bytes, stats, stream, lists, n_binned);
}

int dgmr_splat_backward(const dgmr_gaussians* g, const dgmr_camera* cam, const dgmr_tiling* tiling, const dgmr_splat_geometry* geom,
    const dgmr_binning* bins, int64_t n_pairs, const float* framebuffer, const float* final_transmittance, const float* grad_framebuffer,
    float* screen_grads, float* grad_means, float* grad_scales, float* grad_rotations, float* grad_opacity, float* grad_sh, dgmr_stream stream)
{
    DGMR_ARG_CHECK(g && cam && geom && bins && framebuffer && final_transmittance && grad_framebuffer && screen_grads, "dgmr_splat_backward: null argument");
    DGMR_ARG_CHECK(grad_means && grad_scales && grad_rotations && grad_opacity && grad_sh, "dgmr_splat_backward: null gradient output");
    DGMR_ARG_CHECK(g->dtype == DGMR_F32, "dgmr_splat_backward: the splatter computes in float32");
    DGMR_ARG_CHECK(valid_tiling(tiling), "dgmr_splat_backward: bad tiling");
    DGMR_ARG_CHECK(g->sh_coeffs >= 1 && g->sh_coeffs <= 16 && g->sh_degree >= 0 && g->sh_degree <= 3, "dgmr_splat_backward: bad SH layout");
    const int64_t n = g->n;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (n == 0)
        return DGMR_OK;
    const DevCamera<float> dc = make_dev_camera<float>(*cam, *tiling);
    const int64_t n_tiles = int64_t(dc.grid_x) * dc.grid_y;
    DGMR_HIP_CHECK(hipMemsetAsync(screen_grads, 0, size_t(n) * 9 * sizeof(float), st));
    if (n_pairs > 0) {
        StageScope sc("splat.blend_backward", st, 40.0 * double(n_pairs) + 28.0 * double(int64_t(cam->width) * cam->height) + 8.0 * double(n_tiles));
        splat_blend_backward(*tiling, int(n_tiles), n_pairs, st, bins->ranges, bins->point_list, geom->xy, geom->conic_opacity, geom->rgb, cam->width,
            cam->height, dc.grid_x, cam->background, framebuffer, final_transmittance, grad_framebuffer, screen_grads);
        DGMR_HIP_CHECK(hipGetLastError());
    }
    StageScope sc("splat.preprocess_backward", st, double(n) * (2.0 * (44.0 + 12.0 * g->sh_coeffs) + 59.0));
    k_splat_preprocess_backward<<<unsigned(ceil_div64(n, kPreThreads)), kPreThreads, 0, st>>>(n, make_params(g), dc, geom->tiles_touched,
        reinterpret_cast<const float4*>(geom->conic_opacity), geom->rgb_clamped, screen_grads, grad_means, grad_scales, grad_rotations,
        grad_opacity, grad_sh);
    DGMR_HIP_CHECK(hipGetLastError());
    return DGMR_OK;
}

int dgmr_sort_workspace_size(int64_t n, size_t* bytes)
{
    DGMR_ARG_CHECK(bytes && n >= 0 && n <= int64_t(UINT32_MAX), "dgmr_sort_workspace_size: n out of range");
    *bytes = radix_scratch_bytes(std::max<int64_t>(n, 1));
    return DGMR_OK;
}

int dgmr_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, int64_t n, int32_t begin_bit, int32_t end_bit,
    void* ws, size_t ws_bytes, dgmr_stream stream)
{
    DGMR_ARG_CHECK(n >= 0 && n <= int64_t(UINT32_MAX), "dgmr_sort_pairs: n out of range");
    DGMR_ARG_CHECK(begin_bit >= 0 && end_bit <= 32 && begin_bit <= end_bit, "dgmr_sort_pairs: bits must satisfy 0 <= begin <= end <= 32");
    if (n == 0 || begin_bit == end_bit)
        return DGMR_OK;
    DGMR_ARG_CHECK(keys && vals && keys_tmp && vals_tmp && ws, "dgmr_sort_pairs: null buffer");
    DGMR_ARG_CHECK(ws_bytes >= radix_scratch_bytes(n), "dgmr_sort_pairs: workspace too small");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const SortBuffers buf { keys, vals, keys_tmp, vals_tmp };
    DGMR_HIP_CHECK(radix_sort_pairs(buf, n, nullptr, begin_bit, end_bit, ws, st));
    if (radix_passes(begin_bit, end_bit) % 2 == 1) {
        DGMR_HIP_CHECK(hipMemcpyAsync(keys, keys_tmp, size_t(n) * 4, hipMemcpyDeviceToDevice, st));
        DGMR_HIP_CHECK(hipMemcpyAsync(vals, vals_tmp, size_t(n) * 4, hipMemcpyDeviceToDevice, st));
    }
    return DGMR_OK;
}

int dgmr_scan_workspace_size(int64_t n, size_t* bytes)
{
    DGMR_ARG_CHECK(bytes && n >= 0, "dgmr_scan_workspace_size: n out of range");
    *bytes = scan_scratch_bytes(n);
    return DGMR_OK;
}

int dgmr_scan_u32(const uint32_t* in, uint32_t* out, uint32_t* total, int64_t n, int32_t inclusive, void* ws, size_t ws_bytes,
    dgmr_stream stream)
{
    DGMR_ARG_CHECK(n >= 0, "dgmr_scan_u32: n out of range");
    DGMR_ARG_CHECK(n == 0 || (in && out && ws), "dgmr_scan_u32: null buffer");
    DGMR_ARG_CHECK(ws_bytes >= scan_scratch_bytes(n), "dgmr_scan_u32: workspace too small");
    DGMR_HIP_CHECK(scan_u32(in, out, total, n, inclusive != 0, ws, reinterpret_cast<hipStream_t>(stream)));
    return DGMR_OK;
}

int dgmr_selftest_wave_sum(const float* in, float* out, dgmr_stream stream)
{
    DGMR_ARG_CHECK(in && out, "dgmr_selftest_wave_sum: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    k_selftest_wave_sum<<<1, 64, 0, st>>>(in, out);
    DGMR_HIP_CHECK(hipGetLastError());
    return DGMR_OK;
}

} // extern "C"
