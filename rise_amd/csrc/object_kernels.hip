// object_kernels.hip -- batch closest-hit and any-hit kernels over a scene of
// objects with transforms (object_trace.h).  Persistent waves, one ray per
// lane at a time: each lane's query is in one of three phases (the world tree,
// an object's tree, the top-level walk between them), a wave runs the phases of
// enough lanes in each round, and a lane takes a new ray when its query ends.
// The node-group stack is in LDS when the trees are shallow enough, else in a
// private array.
#include "object_kernels.h"

#include "object_trace.h"
#include "wave_fetch.h"

#include <algorithm>

namespace rise_hip {

namespace {

constexpr int kObjBlock = 128;

// Idle lanes at which a wave takes new rays, and waiting candidates at which it
// certifies them.  A ray's walk over several trees is long, and 500,000 rays
// are two or three a lane, so lanes are not left idle: 500,000 rays into 16
// objects took 2041 us at 20 idle lanes, 2004 at 14, 1980 at 8; 1926 / 1899 /
// 1867 / 1862 at 1 / 2 / 4 / 8 waiting candidates.  Few rays are bound by the
// longest ray's chain and take the large stack's form: 2000 rays 1174 us at 8,
// 1157 at 2 (obj_certify).
constexpr int kRefill = 8;
constexpr int kRefillAny = 20;  // any-hit queries

__device__ inline void load_ray6(const float* __restrict__ rays, int64_t n, int64_t i, float ray[6])
{
#pragma unroll
    for (int k = 0; k < 6; ++k) ray[k] = rays[(int64_t)k * n + i];
}

// The node-group stack: LDS entries per lane when the scene's trees fit into
// kObjLds of them, else a private array (0).  Closest hits of more rays than the
// lanes that are resident so (three waves per SIMD) take kObjLdsSmall entries
// where those are enough: LDS and, with some spills, registers for four waves.
// Records of 30,000 / 200,000 / 500,000 / 1,000,000 rays: 484 / 1382 / 4773 /
// 15,376 us before, 505 / 1270 / 3530 / 11,030 with four waves, 442 us for the
// 30,000 with three (by the rule and with waiting candidates' walks standing
// still 461 / 1183 / 3246 / 10,202).  Any-hit queries lose by it (200,000 rays 430
// -> 484 us) and keep three.
constexpr int kObjLdsSmall = 16, kObjLds = 24;
constexpr int obj_certify(int stack) { return stack == kObjLdsSmall ? 8 : 2; }
constexpr int obj_waves(int stack) { return stack == kObjLdsSmall ? 4 : 1; }

template <int STACK>
struct StackOf {
    using type = ObjLdsStack<STACK>;
};
template <>
struct StackOf<0> {
    using type = ObjStack;
};

template <int STACK>
__device__ inline typename StackOf<STACK>::type make_stack(uint2* lds)
{
    if constexpr (STACK > 0) {
        return ObjLdsStack<STACK>{lds + threadIdx.x, kObjBlock, 0, 0, false};
    } else {
        ObjStack st;
        st.sp = st.base = 0;
        st.overflow = false;
        return st;
    }
}

// Which phases a wave runs in this round: those of at least a kVote-th of its
// busy lanes, so that no phase's code runs for few of them; the others' lanes
// wait until they are more, or the rest is done.  One of the three always has a
// third of the lanes.  500,000 rays into 16 objects: 2178 us with every phase of
// every lane in each round and candidates certified one by one; 2225 / 2076 /
// 2039 / 2032 at a third / quarter / eighth / sixteenth, the last two with the
// refill line at 20 and 14.  (Any-hit queries step every phase in each round:
// with votes 2,000,000 limited shadow rays take 3279 us instead of 2472.)
constexpr int kVote = 8;
struct PhaseVote {
    int n;  // busy lanes
    bool world, object, next;
    __device__ inline explicit PhaseVote(int phase)
    {
        const int w = __popcll(__ballot(phase == kObjPhaseWorld)), o = __popcll(__ballot(phase == kObjPhaseObject));
        n = __popcll(__ballot(phase != kObjPhaseDone));
        world = w * kVote >= n;
        object = o * kVote >= n;
        next = (n - w - o) * kVote >= n;
    }
};

__global__ void reset_fetch(unsigned long long* c) { *c = 0ull; }

// A query's result staged in its rise_hip_hit slot until object_records
// turns it into the record (keeps the record's double arithmetic out of the
// traversal loop's registers).
static_assert(sizeof(ObjectHit) <= sizeof(rise_hip_hit) && alignof(ObjectHit) <= alignof(rise_hip_hit),
              "an ObjectHit must fit in a hit record's slot");

// Persistent: the grid is sized to the resident waves, each lane's first ray
// is assigned statically and later ones are fetched wave-wide (ItemFetch) as
// lanes finish; a query that has ended is written out when its wave fetches.
// REC: stage the ObjectHit in hits[ray] for object_records; else write prim_id
// and t (float world range).
template <int A, bool REC, int STACK>
__global__ __launch_bounds__(kObjBlock, obj_waves(STACK)) void closest_objects(
    ObjectSceneView sc, const float* __restrict__ rays, int64_t n, unsigned faces, int32_t* __restrict__ prim_id,
    float* __restrict__ t_out, rise_hip_hit* __restrict__ hits, unsigned long long* next)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kObjBlock : 1];
    auto st = make_stack<STACK>(lds);
    ObjClosestQuery<A> Q;
    ItemFetch fetch(grid_items(next, n));
    long long ray = -1;
    Q.phase = kObjPhaseDone;
    Q.s.pend = kNoLeaf;
    for (;;) {
        const bool busy = Q.phase != kObjPhaseDone;
        const unsigned long long bm = __ballot(busy);
        if (bm == 0ull || (fetch.more && __popcll(bm) <= 64 - kRefill)) {
            if (!busy && ray >= 0) {
                if (REC) {
                    *reinterpret_cast<ObjectHit*>(hits + ray) = Q.h;
                } else {
                    prim_id[ray] = Q.h.prim_id;
                    t_out[ray] = Q.h.prim_id >= 0 ? (float)Q.h.range : INFINITY;
                }
                ray = -1;
            }
            if (fetch.more) {
                const long long got = fetch.take(busy);
                if (got >= 0) {
                    float r6[6];
                    load_ray6(rays, n, got, r6);
                    objects_closest_begin(sc, r6, st, Q);
                    ray = got;
                }
            } else if (bm == 0ull) {
                break;
            }
        }
        const PhaseVote vote(Q.phase);
        if (vote.world && Q.phase == kObjPhaseWorld) objects_closest_world<true>(sc, faces, st, Q);
        if (vote.object && Q.phase == kObjPhaseObject) objects_closest_object<true>(faces, st, Q);
        const bool waits = (Q.phase == kObjPhaseWorld || Q.phase == kObjPhaseObject) && Q.s.pend != kNoLeaf;
        const int waiting = __popcll(__ballot(waits));
        if (waiting >= obj_certify(STACK) || waiting * 8 >= vote.n) {
            if (waits) objects_closest_commit(sc, Q);
        }
        if (vote.next && Q.phase != kObjPhaseWorld && Q.phase != kObjPhaseObject && Q.phase != kObjPhaseDone)
            objects_closest_next(sc, st, Q);
    }
}

// The intersection record of each ray from its staged ObjectHit, in place.
template <int A>
__global__ __launch_bounds__(kObjBlock) void object_records(ObjectSceneView sc, const float* __restrict__ rays,
                                                            int64_t n, rise_hip_hit* __restrict__ hits)
{
    const int64_t i = (int64_t)blockIdx.x * kObjBlock + threadIdx.x;
    if (i >= n) return;
    const ObjectHit h = *reinterpret_cast<const ObjectHit*>(hits + i);
    float r6[6];
    load_ray6(rays, n, i, r6);
    rise_hip_hit rec;
    objects_record<A>(sc, r6, h, rec);
    hits[i] = rec;
}

template <int A, int STACK>
__global__ __launch_bounds__(kObjBlock) void any_objects(ObjectSceneView sc, const float* __restrict__ rays,
                                                         const float* __restrict__ tmax, int64_t n, unsigned faces,
                                                         uint8_t* __restrict__ occluded, unsigned long long* next)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kObjBlock : 1];
    auto st = make_stack<STACK>(lds);
    ObjAnyQuery<A> Q;
    ItemFetch fetch(grid_items(next, n));
    long long ray = -1;
    bool busy = false;
    for (;;) {
        if (busy) busy = objects_any_step(sc, st, Q);
        const unsigned long long bm = __ballot(busy);
        if (bm != 0ull && !(fetch.more && __popcll(bm) <= 64 - kRefillAny)) continue;
        if (!busy && ray >= 0) {
            occluded[ray] = Q.hit ? 1 : 0;
            ray = -1;
        }
        if (fetch.more) {
            const long long got = fetch.take(busy);
            if (got >= 0) {
                float r6[6];
                load_ray6(rays, n, got, r6);
                objects_any_begin(sc, r6, tmax ? (double)tmax[got] : kRiseInfinity, faces, st, Q);
                ray = got;
                busy = true;
            }
        } else if (bm == 0ull) {
            break;
        }
    }
}

inline unsigned obj_grid(int64_t n) { return (unsigned)((n + kObjBlock - 1) / kObjBlock); }

// Workgroups that fill the device once (resident blocks per CU x CUs), or
// fewer when there are fewer rays.
template <class K>
unsigned resident_grid(K kernel, int64_t n)
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kObjBlock, 0) != hipSuccess || per_cu <= 0)
        per_cu = 2;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((int64_t)cus * per_cu, (int64_t)obj_grid(n)));
}

}  // namespace

hipError_t launch_closest_objects(const ObjectSceneView& sc, int arith, int stack_need, const float* rays, int64_t n,
                                  unsigned faces, int32_t* prim_id, float* t, rise_hip_hit* hits,
                                  unsigned long long* next, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    reset_fetch<<<1, 1, 0, stream>>>(next);
    // The large form's grid serves all its instantiations (each three waves per
    // SIMD), so that only launches of many rays ask for a second one.
    unsigned grid = stack_need <= kObjLds ? resident_grid(closest_objects<kArithIeee, true, kObjLds>, n) : 0u;
    const bool many = stack_need <= kObjLdsSmall && n > (int64_t)kObjBlock * grid;
#define RISE_OBJ_CLOSEST_K(A, R, S)                                                                         \
    do {                                                                                                    \
        if (S != kObjLds) grid = resident_grid(closest_objects<A, R, S>, n);                                \
        closest_objects<A, R, S><<<grid, kObjBlock, 0, stream>>>(sc, rays, n, faces, prim_id, t, hits, next); \
    } while (0)
#define RISE_OBJ_CLOSEST(A, S)                                                                   \
    do {                                                                                         \
        if (hits) {                                                                              \
            RISE_OBJ_CLOSEST_K(A, true, S);                                                      \
            object_records<A><<<obj_grid(n), kObjBlock, 0, stream>>>(sc, rays, n, hits);          \
        } else {                                                                                 \
            RISE_OBJ_CLOSEST_K(A, false, S);                                                     \
        }                                                                                        \
    } while (0)
    if (arith == kArithX86Fma) {
        if (many) RISE_OBJ_CLOSEST(kArithX86Fma, kObjLdsSmall);
        else if (stack_need <= kObjLds) RISE_OBJ_CLOSEST(kArithX86Fma, kObjLds);
        else RISE_OBJ_CLOSEST(kArithX86Fma, 0);
    } else {
        if (many) RISE_OBJ_CLOSEST(kArithIeee, kObjLdsSmall);
        else if (stack_need <= kObjLds) RISE_OBJ_CLOSEST(kArithIeee, kObjLds);
        else RISE_OBJ_CLOSEST(kArithIeee, 0);
    }
#undef RISE_OBJ_CLOSEST
#undef RISE_OBJ_CLOSEST_K
    return hipGetLastError();
}

hipError_t launch_any_objects(const ObjectSceneView& sc, int arith, int stack_need, const float* rays,
                              const float* tmax, int64_t n, unsigned faces, uint8_t* occluded,
                              unsigned long long* next, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    reset_fetch<<<1, 1, 0, stream>>>(next);
#define RISE_OBJ_ANY(A, S)                                                                               \
    any_objects<A, S><<<resident_grid(any_objects<A, S>, n), kObjBlock, 0, stream>>>(sc, rays, tmax, n, faces, \
                                                                                      occluded, next)
    if (arith == kArithX86Fma) {
        if (stack_need <= kObjLds) RISE_OBJ_ANY(kArithX86Fma, kObjLds);
        else RISE_OBJ_ANY(kArithX86Fma, 0);
    } else {
        if (stack_need <= kObjLds) RISE_OBJ_ANY(kArithIeee, kObjLds);
        else RISE_OBJ_ANY(kArithIeee, 0);
    }
#undef RISE_OBJ_ANY
    return hipGetLastError();
}

}  // namespace rise_hip
