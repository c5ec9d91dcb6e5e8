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
// Lanes whose candidate waits when the wave certifies: 2868 us at 1, 2853 at
// 2, 2880 at 4, 2960 at 8 (the waiting rays visit nodes that the hit would
// have culled); with vertex records and any-hit shadows alike 1-2%.
#ifndef RISE_CERTIFY
#define RISE_CERTIFY 2
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

// The next item of every idle lane of a wave (`busy` false), wave-wide: first
// the thread's own (one per thread of the grid), so that a launch starts
// without a burst of atomics on one address, then items of the wave's own
// chunk, claimed from the shared counter (which counts from the grid's size)
// with one atomic per chunk.  Atomics on one address serialize at about 10 ns
// each, so a claim per refill bounds the launch; chunks shrink as the items
// run out (a quarter of an even share, between 32 and RISE_CHUNK), so that
// the waves end together.
struct ItemFetch {
    unsigned long long* next;
    int64_t n;
    unsigned long long cur, end;  // wave-uniform: the claimed items not yet taken
    bool started;
    bool more;  // wave-uniform: the items may not be exhausted

    __device__ inline ItemFetch(unsigned long long* counter, int64_t items)
        : next(counter), n(items), cur(0), end(0), started(false), more(items > 0)
    {
    }
    // Every lane of the wave calls; the lane's new item, or -1.
    __device__ inline long long take(bool busy)
    {
        const unsigned long long first = (unsigned long long)gridDim.x * blockDim.x, total = (unsigned long long)n;
        unsigned long long i;
        if (!started) {
            i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
            more = total > first;
            started = true;
            cur = end = first;
        } else {
            const unsigned long long im = __ballot(!busy);
            const unsigned want = (unsigned)__popcll(im), left = (unsigned)(end - cur);
            const unsigned rank =
                __builtin_amdgcn_mbcnt_hi((unsigned)(im >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)im, 0u));
            i = cur + rank;
            cur += want;
            if (want > left) {
                const float share = (float)(total - end) * 16.0f / (float)first;  // a quarter of this wave's even share
                const unsigned size = (unsigned)fminf(fmaxf(share, 32.0f), (float)RISE_CHUNK);
                const unsigned need = want - left, take = size > need ? size : need;
                unsigned long long base = 0;
                if (__lane_id() == 0) base = atomicAdd(next, (unsigned long long)take);
                const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)base);
                const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(base >> 32));
                base = first + (((unsigned long long)hi << 32) | lo);
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

// Closest-hit queries in persistent waves: each lane steps one query a node at
// a time.  What few lanes need per step is put off until many do:
//   * a query that has ended stays in its lane until RISE_REFILL lanes are
//     idle (or none is busy); then all of them certify what still waits,
//     finish (world range, stores) and take new items together, the new items
//     claimed with one atomic per wave;
//   * candidates that the filter has passed are certified once RISE_CERTIFY
//     lanes, or an eighth of the busy ones, have one (closest_step's DEFER).
// Bound by instruction issue: the kernel's time follows its vector
// instructions (2.15e9 a launch before, 1.9e9 now at 48 of 64 lanes busy).  On
// the 1M-triangle, 6.07M-ray cast 3405 -> 2880 us against one claim per refill,
// certifying and finishing at once, and a node test that branched per child.
// Counted queries (COUNT) certify at once, so that their counts are those of
// the traversal alone, whatever else its wave holds.
// begin(item, r, s) starts a query, or returns false to skip the item;
// finish(item, r, s) takes its result.
template <bool COUNT, bool CULL, bool F64, class R, class Stack, class Begin, class Finish>
__device__ inline void persist_closest(Stack& st, int64_t n, unsigned long long* next, unsigned& nn, unsigned& nt,
                                       const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                       Begin begin, Finish finish)
{
    R r;
    ClosestState s;
    s.pend = kNoLeaf;
    ItemFetch fetch(next, n);
    long long item = -1;
    bool busy = false;
    for (;;) {
        if (busy) busy = closest_step<COUNT, CULL, F64, !COUNT>(r, nodes, tris, st, s, nn, nt, tri64);
        const unsigned long long bm = __ballot(busy);
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
__device__ inline void persist_any(Stack& st, int64_t n, unsigned long long* next, unsigned& nn, unsigned& nt,
                                   const NodeSlot* const& nodes, const Tri48* const& tris, const double* tri64,
                                   Begin begin, Finish finish)
{
    R r;
    AnyState s;
    ItemFetch fetch(next, n);
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
    }
}

}  // namespace rise_hip
