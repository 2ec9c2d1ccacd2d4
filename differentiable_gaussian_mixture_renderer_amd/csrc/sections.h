// SPDX-License-Identifier: GPL-3.0-or-later
// The marcher's sample-section list (reference: src/dgmr/marching_steps.h:28-200).
// Usable on the host as well: the CPU tests run it against the restatement.
#pragma once

#include <cmath>
#include <type_traits>
#include <utility>

#if defined(__HIPCC__)
#define DGMR_SECTIONS_FN __host__ __device__ __forceinline__
#else
#define DGMR_SECTIONS_FN inline
#endif

namespace dgmr {

// f(0), f(1), ... f(N - 1) with compile-time arguments: arrays kept in
// registers are then only ever indexed by constants (a loop that the compiler
// unrolls late leaves them one register tuple, copied at every branch)
template <class F, int... I>
DGMR_SECTIONS_FN void static_for_each(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I> {}), ...);
}
template <int N, class F>
DGMR_SECTIONS_FN void static_for(F&& f)
{
    static_for_each(f, std::make_integer_sequence<int, N> {});
}

template <class S>
struct Section {
    S start, end, dt;
};

namespace sections {

// whether the condition holds on an active lane of the wave (host: one lane)
DGMR_SECTIONS_FN bool any_lane(bool p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(p) != 0;
#else
    return p;
#endif
}

template <class S>
DGMR_SECTIONS_FN S smin(S a, S b) { return b < a ? b : a; }
template <class S>
DGMR_SECTIONS_FN S smax(S a, S b) { return a < b ? b : a; }

} // namespace sections

// A pixel's sections in three planes, interleaved over the NT pixels that share
// the storage: field f of section i is base[(f kSlots + i) NT] (base: this
// pixel's first word, so the lanes of a wave touch consecutive words and the
// three fields of a section share one address).  One section more than the
// list holds: put() writes what falls off the end there.
template <class S, int CAP, int NT>
struct SectionStore {
    static constexpr int kSlots = CAP + 1;
    S* base;
    DGMR_SECTIONS_FN S start(int i) const { return base[i * NT]; }
    DGMR_SECTIONS_FN S end(int i) const { return base[(kSlots + i) * NT]; }
    DGMR_SECTIONS_FN S dt(int i) const { return base[(2 * kSlots + i) * NT]; }
    DGMR_SECTIONS_FN Section<S> get(int i) const { return { start(i), end(i), dt(i) }; }
    DGMR_SECTIONS_FN void set(int i, const Section<S>& v)
    {
        S* p = base + i * NT;
        p[0] = v.start;
        p[kSlots * NT] = v.end;
        p[2 * kSlots * NT] = v.dt;
    }
};

// marching_steps::DensityArray (marching_steps.h:35-200): a sorted list of
// disjoint sections over [start, end) holding the minimum step; when full,
// end() shrinks to the last section's end.
//
// Inserting e keeps the overlapped sections with a smaller step, fills the gaps
// between them with e, and cuts e out of those with a larger step (a section
// of exactly e's step that e overlaps merges with it).  put() does that in one
// pass over the slots in registers: the same selections as the reference's
// in-place merge, no arithmetic, so the same list (sequences of sections with
// equal steps, empty ones or NaN take put_in_order, the reference's own order
// of operations).  Slot blocks before the first and after the last change on
// the wave are skipped or only moved.  VALU and branch bound: about 440 vector
// instructions; the in-order merge, with lane-divergent loops through LDS and a
// ring in private memory, took 10 000 cycles per section and wave where this
// takes 7 500 (200k Gaussians at 1024^2, two waves per SIMD).
template <class S, int CAP, int NT>
struct SectionList {
    SectionStore<S, CAP, NT> data;
    int size;
    S start_, end_;
    bool in_order; // this step's list holds an empty section or a NaN: only put_in_order keeps the reference's list

    DGMR_SECTIONS_FN void reset(S start)
    {
        size = 0;
        start_ = start;
        end_ = S(__builtin_huge_val());
        in_order = false;
    }

    DGMR_SECTIONS_FN int first_ending_after(S v, int from) const
    {
        for (int i = from; i < size; ++i)
            if (data.end(i) > v)
                return i;
        return size;
    }

    DGMR_SECTIONS_FN static void combine(const Section<S>& a, const Section<S>& b, Section<S>* out)
    {
        if (a.start < b.start)
            out[0] = { a.start, sections::smin(a.end, b.start), a.dt };
        else
            out[0] = { b.start, sections::smin(b.end, a.start), b.dt };
        if (b.end < a.end)
            out[2] = { b.end, a.end, a.dt };
        else
            out[2] = { a.end, b.end, b.dt };
        out[1] = { out[0].end, out[2].start, sections::smin(a.dt, b.dt) };
    }

    DGMR_SECTIONS_FN void put(Section<S> e)
    {
        if (e.end <= start_ || e.start >= end_)
            return;
        e.start = sections::smax(start_, e.start);
        e.end = sections::smin(end_, e.end);
        in_order = in_order || !(e.start < e.end) || e.dt != e.dt;
        S a[CAP], b[CAP], d[CAP];
        // the first block of 4 slots that some lane needs: those before it end before e
        int kb = 0;
        static_for<CAP / 4 - 1>([&](auto q) {
            constexpr int k = q + 1;
            if (!sections::any_lane(size < 4 * k || !(data.end(4 * k - 1) <= e.start)))
                kb = k;
        });
        bool equal = false;
        static_for<CAP / 4>([&](auto k) {
            if (k >= kb)
                static_for<4>([&](auto j) {
                    constexpr int i = 4 * k + j;
                    const Section<S> s = data.get(i);
                    a[i] = s.start;
                    b[i] = s.end;
                    d[i] = s.dt;
                });
        });
        static_for<CAP / 4>([&](auto k) {
            if (k >= kb)
                static_for<4>([&](auto j) {
                    constexpr int i = 4 * k + j;
                    equal = equal || (i < size && b[i] > e.start && a[i] < e.end && d[i] == e.dt);
                });
        });
        if (in_order || equal) {
            put_in_order(e);
            return;
        }
        const S s = e.start, t = e.end;
        S p = s;          // where the part of e that is still to be written begins
        int wr = 4 * kb;  // next slot written
        bool fin = false; // e is written up to its end
        bool seen = false, more = true;
        const auto emit = [&](S from, S to, S step) {
            data.set(wr < CAP ? wr : CAP, { from, to, step });
            ++wr;
        };
        static_for<CAP / 4>([&](auto k) {
            if (k >= kb && more) {
                if (!sections::any_lane(!fin)) {
                    // past e on every lane: what is left moves as it is
                    static_for<4>([&](auto j) {
                        constexpr int i = 4 * k + j;
                        if (i < size)
                            emit(a[i], b[i], d[i]);
                    });
                    return;
                }
                static_for<4>([&](auto j) {
                    constexpr int i = 4 * k + j;
                    const bool valid = i < size;
                    const bool after = valid && b[i] > s; // ends after e begins
                    const bool ov = after && a[i] < t;
                    const bool less = d[i] < e.dt;
                    const bool low = ov && less, cut = ov && !less;
                    const bool past = valid && b[i] > t;
                    seen = seen || after;
                    if (cut && a[i] < s)
                        emit(a[i], s, d[i]); // what lies before e
                    // e up to this section, or its last part
                    const S to = low ? a[i] : t;
                    if ((low || (past && !fin)) && p < to)
                        emit(p, to, e.dt);
                    p = low ? b[i] : p;
                    fin = fin || past;
                    // the section itself, or what lies after e
                    if (valid && (!cut || past))
                        emit(cut ? t : a[i], b[i], d[i]);
                });
                // nothing moves any more on any lane
                constexpr int done = 4 * k + 4;
                more = sections::any_lane(!fin || wr != done || size < done);
                if (!more)
                    wr = size;
            }
        });
        if (!fin && p < t)
            emit(p, t, e.dt);
        if (!seen) { // beyond every section: appended as it is, or the list ends there
            if (size < CAP)
                ++size;
            else
                end_ = s;
            return;
        }
        size = wr < CAP ? wr : CAP;
        if (size == CAP)
            end_ = sections::smin(end_, data.end(CAP - 1));
    }

    // the reference's insertion step for step (in-place merge through a small
    // ring buffer); e is clipped to [start_, end_)
    DGMR_SECTIONS_FN void put_in_order(Section<S> e)
    {
        const int first = first_ending_after(e.start, 0);
        if (first >= size) {
            if (first < CAP)
                data.set(size++, e);
            else
                end_ = e.start;
            return;
        }
        int stop = first_ending_after(e.end, first);
        if (stop < size && data.start(stop) < e.end)
            ++stop;
        Section<S> ring[CAP];
        unsigned ring_r = 0, ring_w = 0;
        int rd = first, wr = first, inserted = 0;
        while (rd < stop + inserted && wr < CAP) {
            if (rd < size)
                ring[(ring_w++) % CAP] = data.get(rd++);
            if (ring_r >= ring_w)
                break;
            const Section<S> head = ring[ring_r % CAP];
            if (head.end <= e.start) {
                data.set(wr++, ring[(ring_r++) % CAP]);
                continue;
            }
            if (head.start >= e.end)
                break;
            Section<S> parts[3];
            combine(ring[(ring_r++) % CAP], e, parts);
            if (parts[0].dt == parts[1].dt) {
                parts[1].start = parts[0].start;
                parts[0].end = parts[0].start;
            }
            e = parts[2];
            if (parts[0].end - parts[0].start <= 0) {
                if (parts[1].dt == parts[2].dt) {
                    e.start = parts[1].start;
                    continue;
                }
                data.set(wr++, parts[1]);
            } else {
                data.set(wr++, parts[0]);
                if (parts[1].dt == parts[2].dt) {
                    e.start = parts[1].start;
                    continue;
                }
                ++inserted;
                ring[(--ring_r) % CAP] = parts[1];
            }
        }
        if (e.end - e.start > 0 && wr < CAP) {
            if (rd < size)
                ring[(ring_w++) % CAP] = data.get(rd++);
            data.set(wr++, e);
        }
        while (ring_w - ring_r && wr < CAP) {
            if (rd < size)
                ring[(ring_w++) % CAP] = data.get(rd++);
            data.set(wr++, ring[(ring_r++) % CAP]);
        }
        size = wr + size - rd;
        if (size == CAP)
            end_ = sections::smin(end_, data.end(size - 1));
    }
};

} // namespace dgmr
