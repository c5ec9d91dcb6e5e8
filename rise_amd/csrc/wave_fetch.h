// wave_fetch.h -- wave-wide dynamic work fetch for persistent traversal kernels.
#pragma once

#include "trace_core.h"

#include <hip/hip_runtime.h>

#include <cstdint>

// Idle lanes at which a wave fetches new items: closest-hit and any-hit
// queries.  A fetch costs some 700 instructions whatever the lanes it serves
// (the new rays' double square root and division, the finished ones' world
// range), so lanes wait for company: closest-hit ray cast of 6.07M rays
// 2886 us at 20, 2896 at 14, 2902 at 28, 2966 at 36; 12 batched renders
// (shadow rays) 46.1 ms at 22-28, 47.1 ms at 34.
#ifndef RISE_REFILL
#define RISE_REFILL 20
#endif
#ifndef RISE_REFILL_ANY
#define RISE_REFILL_ANY 28
#endif
// Items of one claim, at most (ItemFetch): 64 items make the same ray cast
// 2942 us, 256 and 512 2880.
#ifndef RISE_CHUNK
#define RISE_CHUNK 256
#endif
// Lanes whose candidate waits when the wave certifies, the others going on: the
// ray cast takes 2924 us at 1, 2848 at 2, 2803 at 4, 2790 at 8.
#ifndef RISE_CERTIFY
#define RISE_CERTIFY 8
#endif

namespace rise_hip {

template <int STACK>
struct StackKind {
    using type = LdsStack<STACK>;
};
template <>
struct StackKind<0> {
    using type = PrivStack;
};

// This lane's empty node-group stack: STACK entries of `lds` strided by the
// workgroup size, or (STACK 0) a private array.
template <int STACK>
__device__ inline typename StackKind<STACK>::type make_stack(uint2* lds, int stride)
{
    typename StackKind<STACK>::type st;
    if constexpr (STACK > 0) {
        st.base = lds + threadIdx.x;
        st.stride = stride;
    }
    st.sp = 0;
    return st;
}

// Lanes that share one ray once few rays are left in a wave (coop_* below).
constexpr int kCoopLanes = 8, kCoopRays = 64 / kCoopLanes;

// Where a launch's items come from: `total` of them, the first `first` assigned
// to the threads statically (thread `self` of them), the others claimed from
// `next` (which counts from `first`).  per_wave < 64: each wave takes only that
// many of its first items, its lowest lanes one each, and the launch has no
// others.
struct ItemSource {
    unsigned long long* next;
    unsigned long long total, first, self;
    int per_wave;
};

// All items of a grid-wide launch.
__device__ inline ItemSource grid_items(unsigned long long* next, int64_t n)
{
    return ItemSource{next, n > 0 ? (unsigned long long)n : 0ull, (unsigned long long)gridDim.x * blockDim.x,
                      (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x, 64};
}

// A grid-wide launch of kCoopRays items a wave.
__device__ inline ItemSource sparse_items(int64_t n)
{
    const unsigned long long wave = ((unsigned long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    return ItemSource{nullptr, n > 0 ? (unsigned long long)n : 0ull, n > 0 ? (unsigned long long)n : 0ull,
                      wave * kCoopRays + __lane_id(), kCoopRays};
}

// n items of one workgroup of BLOCK threads: an even share for every wave while
// there are at most BLOCK, so that no wave has more rays than it must; else
// one a thread and the others from `next` (LDS, cleared).
template <int BLOCK>
__device__ inline ItemSource block_items(unsigned long long* next, unsigned n)
{
    const unsigned wave = threadIdx.x >> 6;
    if (n > (unsigned)BLOCK) return ItemSource{next, n, (unsigned long long)BLOCK, threadIdx.x, 64};
    const unsigned share = (n + BLOCK / 64 - 1) / (BLOCK / 64);
    return ItemSource{nullptr, n, n, (unsigned long long)(wave * share + __lane_id()), (int)share};
}

// The next item of every idle lane of a wave (`busy` false), wave-wide: first
// the thread's own, so that a launch starts without a burst of atomics on one
// address, then items of the wave's own chunk, claimed from the shared counter
// with one atomic per chunk.  Atomics on one address serialize at about 10 ns
// each, so a claim per refill bounds the launch; chunks shrink as the items
// run out (a quarter of an even share, between 32 and RISE_CHUNK), so that
// the waves end together.
struct ItemFetch {
    ItemSource src;
    unsigned long long cur, end;  // wave-uniform: the claimed items not yet taken
    bool started;
    bool more;  // wave-uniform: the items may not be exhausted

    __device__ inline explicit ItemFetch(const ItemSource& s)
        : src(s), cur(0), end(0), started(false), more(s.total > 0)
    {
    }
    // Every lane of the wave calls; the lane's new item, or -1.
    __device__ inline long long take(bool busy)
    {
        const unsigned long long total = src.total;
        unsigned long long i;
        if (!started) {
            i = (int)__lane_id() < src.per_wave ? src.self : total;
            more = total > src.first;
            started = true;
            cur = end = src.first;
        } else {
            const unsigned long long im = __ballot(!busy);
            const unsigned want = (unsigned)__popcll(im), left = (unsigned)(end - cur);
            const unsigned rank =
                __builtin_amdgcn_mbcnt_hi((unsigned)(im >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)im, 0u));
            i = cur + rank;
            cur += want;
            if (want > left) {
                // A quarter of this wave's even share.
                const float share = (float)(total - end) * 16.0f / (float)src.first;
                const unsigned size = (unsigned)fminf(fmaxf(share, 32.0f), (float)RISE_CHUNK);
                const unsigned need = want - left, take = size > need ? size : need;
                unsigned long long base = 0;
                if (__lane_id() == 0) base = atomicAdd(src.next, (unsigned long long)take);
                const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)base);
                const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(base >> 32));
                base = src.first + (((unsigned long long)hi << 32) | lo);
                if (rank >= left) i = base + (rank - left);
                cur = base + need;
                end = base + take;
                if (end > total) end = total;
            }
            more = cur < end || end < total;
        }
        return !busy && i < total ? (long long)i : -1;
    }
};

// ---- one ray over eight lanes -------------------------------------------------
//
// Once a wave has at most kCoopRays rays left and none to fetch, each ray gets
// kCoopLanes lanes: lane j of a group tests slot j ^ oinv of the ray's next
// node, so one ballot gives every group its hit mask in visiting order, and the
// lanes of accepted leaves filter their triangles side by side.  A step is some
// 120 instructions instead of 400, and what bounds the end of a launch (or a
// launch of few rays) is the longest ray's chain of steps: 7072 rays into 20,000
// triangles 107 -> 68 us, a million shadow rays into 200,000 574 -> 544 us (and
// the additional code costs launches with no short end 0.5%: six million rays
// into a million triangles 2836 -> 2850 us).

__device__ inline long long shfl_i64(long long v, int src)
{
    const unsigned lo = (unsigned)__shfl((int)(unsigned)v, src), hi = (unsigned)__shfl((int)(unsigned)(v >> 32), src);
    return (long long)(((unsigned long long)hi << 32) | lo);
}
__device__ inline double shfl_f64(double v, int src)
{
    return __builtin_bit_cast(double, shfl_i64(__builtin_bit_cast(long long, v), src));
}

// This lane's group's ray: the lane that holds it (the group-th busy lane of
// bm), -1 for a group without one.
__device__ inline int coop_owner(unsigned long long bm)
{
    const int group = (int)__lane_id() / kCoopLanes;
    for (int k = 0; k < group; ++k) bm &= bm - 1ull;
    return bm ? __builtin_ctzll(bm) : -1;
}

// One node visit of a group: like visit_node, with the group's lanes at its
// slots.  leaf, count: the triangles of this lane's accepted leaf (count 0:
// none).  Every lane of the wave calls; `on`: its group's ray goes on.
template <class Stack, class R>
__device__ inline void coop_visit(bool on, const R& r, const NodeSlot* __restrict__ nodes, Stack& st, NodeGroup& g,
                                  float pad_limit, unsigned& leaf, unsigned& count)
{
    bool internal = false;
    unsigned base = 0, imask = 0;
    count = 0;
    leaf = 0;
    if (on) {
        const unsigned k = __builtin_ctz(g.hits);
        g.hits &= g.hits - 1u;
        const unsigned at = k ^ r.oinv;
        const unsigned ni = g.base + __builtin_popcount(g.imask & ((1u << at) - 1u));
        // Every lane of the group writes the same entry.
        if (g.hits) st.push(make_uint2(g.base, g.hits | (g.imask << 8)));
        const unsigned char* node = reinterpret_cast<const unsigned char*>(nodes + ni);
        const unsigned slot = (__lane_id() & (kCoopLanes - 1)) ^ r.oinv;
        const uint4 w0 = *reinterpret_cast<const uint4*>(node);
        const uint2 w1 = *reinterpret_cast<const uint2*>(node + 16);
        const unsigned meta = node[24 + slot];
        const bool hit = meta != 0u && slot_accepted(r, node, w0, slot, pad_limit);
        imask = (w0.w >> 24) & 0xffu;
        base = w1.x;
        internal = hit && ((imask >> slot) & 1u);
        if (hit && !internal) {
            count = meta >> 5;
            leaf = w1.y + (meta & 31u);
        }
    }
    const unsigned long long im = __ballot(internal);
    if (on) g = NodeGroup{base, (unsigned)(im >> (__lane_id() & ~(unsigned)(kCoopLanes - 1))) & 0xffu, imask};
}

// The rays of the busy lanes bm (at most kCoopRays) traced to their ends by
// kCoopLanes lanes each.  Every lane of the wave calls, with its query's state;
// no candidate waits.  `lds`: the workgroup's node-group stacks.
template <bool CULL, bool F64, int STACK, class R, class Begin, class Finish>
__device__ inline void coop_closest(unsigned long long bm, long long item, R& r, ClosestState& s, LdsStack<STACK>& st,
                                    const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                    Begin begin, Finish finish)
{
    const int owner = coop_owner(bm), from = owner < 0 ? 0 : owner;
    bool on = owner >= 0;
    item = shfl_i64(item, from);
    ClosestState h;
    h.g = NodeGroup{(unsigned)__shfl((int)s.g.base, from), (unsigned)__shfl((int)s.g.hits, from),
                    (unsigned)__shfl((int)s.g.imask, from)};
    h.best_leaf = (unsigned)__shfl((int)s.best_leaf, from);
    h.best_id = __shfl(s.best_id, from);
    h.tlim = __shfl(s.tlim, from);
    h.best_t = shfl_f64(s.best_t, from);
    const int sp = __shfl(st.sp, from);
    LdsStack<STACK> gst = st;  // the owner's stack
    gst.base = st.base + (from - (int)__lane_id());
    gst.sp = sp;
    if (on) begin(item, r, s);
    s.g = h.g;
    s.best_leaf = h.best_leaf;
    s.best_id = h.best_id;
    s.tlim = h.tlim;
    s.best_t = h.best_t;
    while (__ballot(on) != 0ull) {
        unsigned leaf, count;
        coop_visit(on, r, nodes, gst, s.g, s.tlim, leaf, count);
        // The lane's triangles that pass with the best hit before this node; then
        // the group's, one after the other in the order of a single lane's walk
        // (slots, their triangles), each in all lanes of the group alike: the
        // range test again once another has been certified, and the certifier.
        unsigned passed = 0;
        float t;
        for (unsigned k = 0; k < count; ++k)
            if (passes_filter<CULL, F64, false>(r, tris, tri64, leaf + k, s.faces, (float)s.best_t, t))
                passed |= 1u << k;
        const unsigned lane0 = __lane_id() & ~(unsigned)(kCoopLanes - 1);
        bool first = true;
        unsigned long long pm = __ballot(passed != 0u);
        while (pm != 0ull) {
            const unsigned gm = (unsigned)(pm >> lane0) & 0xffu;
            const unsigned at = gm ? lane0 + (__builtin_ctz(xor_permute8(gm, r.oinv)) ^ r.oinv) : __lane_id();
            // A leaf holds at most seven, so bit 7 stands for none.
            const unsigned next = (unsigned)__shfl((int)(leaf + __builtin_ctz(passed | 0x80u)), (int)at);
            if (at == __lane_id()) passed &= passed - 1u;
            pm = __ballot(passed != 0u);
            if (gm) {
                if (first || passes_filter<CULL, F64, false>(r, tris, tri64, next, s.faces, (float)s.best_t, t)) {
                    s.pend = next;
                    closest_commit<F64>(r, tris, tri64, s);
                }
                first = false;
            }
        }
        if (on && !next_group(gst, s.g)) {
            if ((__lane_id() & (kCoopLanes - 1)) == 0) finish(item, r, s);
            on = false;
        }
    }
}

// The same for any-hit queries: a group is done once one of its lanes
// certifies a triangle within range.
template <bool CULL, bool F64, int STACK, class R, class Begin, class Finish>
__device__ inline void coop_any(unsigned long long bm, long long item, R& r, AnyState& s, LdsStack<STACK>& st,
                                const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                Begin begin, Finish finish)
{
    const int owner = coop_owner(bm), from = owner < 0 ? 0 : owner;
    bool on = owner >= 0;
    item = shfl_i64(item, from);
    const NodeGroup g{(unsigned)__shfl((int)s.g.base, from), (unsigned)__shfl((int)s.g.hits, from),
                      (unsigned)__shfl((int)s.g.imask, from)};
    const int sp = __shfl(st.sp, from);
    LdsStack<STACK> gst = st;
    gst.base = st.base + (from - (int)__lane_id());
    gst.sp = sp;
    if (on) begin(item, r, s);
    s.g = g;
    while (__ballot(on) != 0ull) {
        unsigned leaf, count;
        coop_visit(on, r, nodes, gst, s.g, s.tlim, leaf, count);
        bool hit = false;
        for (; count && !hit; --count, ++leaf) {
            float t;
            if (!passes_filter<CULL, F64, true>(r, tris, tri64, leaf, s.faces, s.fbest, t)) continue;
            s.pend = leaf;
            any_commit<F64>(r, tris, tri64, s);
            hit = s.hit;
        }
        const unsigned long long hm = __ballot(on && hit);
        if (on) {
            s.hit = ((hm >> (__lane_id() & ~(unsigned)(kCoopLanes - 1))) & 0xffull) != 0ull;
            if (s.hit || !next_group(gst, s.g)) {
                if ((__lane_id() & (kCoopLanes - 1)) == 0) finish(item, s);
                on = false;
            }
        }
    }
}

template <class Stack>
struct CoopStack {
    static constexpr bool value = false;  // a private array cannot be read by other lanes
};
template <int STACK>
struct CoopStack<LdsStack<STACK>> {
    static constexpr bool value = true;
};

// Closest-hit queries in persistent waves: each lane steps one query a node at
// a time.  What few lanes need per step is put off until many do:
//   * a query that has ended stays in its lane until RISE_REFILL lanes are
//     idle (or none is busy); then all of them certify what still waits,
//     finish (world range, stores) and take new items together, the new items
//     claimed with one atomic per wave;
//   * a candidate that the filter has passed waits, and its query with it, until
//     RISE_CERTIFY lanes, or an eighth of the busy ones, have one
//     (closest_step's DEFER).
// Bound by instruction issue: the kernel's time follows its vector
// instructions, 2.03e9 a launch of the 1M-triangle, 6.07M-ray cast with 35 of 64
// lanes active in one (2.31e9 with one claim per refill, certifying and finishing
// at once, and a node test that branched per child: 3405 us, 2790 now).
// Counted queries (COUNT) certify at once; their counts and hits are the same.
// begin(item, r, s) starts a query, or returns false to skip the item;
// finish(item, r, s) takes its result.
template <bool COUNT, bool CULL, bool F64, class R, class Stack, class Begin, class Finish>
__device__ inline void persist_closest(Stack& st, const ItemSource& items, unsigned& nn, unsigned& nt,
                                       const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                       Begin begin, Finish finish)
{
    R r;
    ClosestState s;
    s.pend = kNoLeaf;
    ItemFetch fetch(items);
    long long item = -1;
    bool busy = false;
    for (;;) {
        if (busy) busy = closest_step<COUNT, CULL, F64, !COUNT>(r, nodes, tris, st, s, nn, nt, tri64);
        const unsigned long long bm = __ballot(busy);
        if constexpr (CoopStack<Stack>::value && !COUNT) {
            if (!fetch.more && bm != 0ull && __popcll(bm) <= kCoopRays) {
                if (item >= 0 && s.pend != kNoLeaf) closest_commit<F64>(r, tris, tri64, s);
                if (!busy && item >= 0) finish(item, r, s);
                coop_closest<CULL, F64>(bm, item, r, s, st, nodes, tris, tri64, begin, finish);
                break;
            }
        }
        if (bm == 0ull || (fetch.more && __popcll(bm) <= 64 - RISE_REFILL)) {
            if (!busy && item >= 0) {
                if (s.pend != kNoLeaf) closest_commit<F64>(r, tris, tri64, s);
                finish(item, r, s);
                item = -1;
            }
            if (fetch.more) {
                const long long got = fetch.take(busy);
                if (got >= 0) {
                    st.sp = 0;
                    busy = begin(got, r, s);
                    if (busy) item = got;
                }
            } else if (bm == 0ull) {
                break;
            }
        } else {
            const int waiting = __popcll(__ballot(busy && s.pend != kNoLeaf));
            if ((waiting >= RISE_CERTIFY || waiting * 8 >= __popcll(bm)) && busy && s.pend != kNoLeaf)
                closest_commit<F64>(r, tris, tri64, s);
        }
    }
}

// Any-hit queries in persistent waves.  A query stops at the first candidate
// that the filter passes (nearly all of them are hits) and is certified with
// the other idle lanes' when the wave refills, or, once no items are left to
// fetch, when a quarter as many wait as are busy; one that fails goes on.
template <bool COUNT, bool CULL, bool F64, class R, class Stack, class Begin, class Finish>
__device__ inline void persist_any(Stack& st, const ItemSource& items, unsigned& nn, unsigned& nt,
                                   const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                   Begin begin, Finish finish)
{
    R r;
    AnyState s;
    ItemFetch fetch(items);
    long long item = -1;
    bool busy = false;
    for (;;) {
        if (busy) busy = any_step<COUNT, CULL, F64, !COUNT>(r, nodes, tris, st, s, nn, nt, tri64);
        const unsigned long long bm = __ballot(busy);
        bool now = bm == 0ull;
        if (fetch.more) now = now || __popcll(bm) <= 64 - RISE_REFILL_ANY;
        else now = now || 4 * __popcll(__ballot(!busy && item >= 0 && !s.hit && !s.over)) >= __popcll(bm);
        if (now) {
            if (!busy && item >= 0) {
                if (!s.hit && s.pend != kNoLeaf) any_commit<F64>(r, tris, tri64, s);
                if (s.hit || s.over) {
                    finish(item, s);
                    item = -1;
                } else {
                    busy = true;
                }
            }
            if (fetch.more) {
                const long long got = fetch.take(busy);
                if (got >= 0) {
                    st.sp = 0;
                    busy = begin(got, r, s);
                    if (busy) item = got;
                }
            } else if (__ballot(busy) == 0ull) {
                break;
            }
        }
        if constexpr (CoopStack<Stack>::value && !COUNT) {
            // Few rays left and none to fetch: first certify what waits.
            if (!fetch.more && __popcll(__ballot(item >= 0)) <= kCoopRays) {
                if (!busy && item >= 0) {
                    if (!s.hit && s.pend != kNoLeaf) any_commit<F64>(r, tris, tri64, s);
                    if (s.hit || s.over) {
                        finish(item, s);
                        item = -1;
                    } else {
                        busy = true;
                    }
                }
                const unsigned long long left = __ballot(busy);
                if (left != 0ull) coop_any<CULL, F64>(left, item, r, s, st, nodes, tris, tri64, begin, finish);
                break;
            }
        }
    }
}

}  // namespace rise_hip
