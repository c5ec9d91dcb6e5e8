// trace_kernels.hip -- batch closest-hit and any-hit kernels over a ray SoA.
//
// These replace the per-ray IObjectManager::IntersectRay / IntersectShadowRay
// calls (Interfaces/IObjectManager.h:38-68, Managers/ObjectManager.cpp:270-373)
// with one launch over a whole batch.  One lane per ray, eight where few
// rays are left or given (wave_fetch.h); the node-group stack lives in LDS (8
// or 16 entries per lane) when the tree is shallow enough, else in a private
// array.
#include "rise_hip.h"
#include "trace_core.h"
#include "trace_kernels.h"
#include "wave_fetch.h"

#include <algorithm>
#include <mutex>

namespace rise_hip {

static_assert(kArithIeee == RISE_HIP_ARITH_IEEE && kArithX86Fma == RISE_HIP_ARITH_X86_FMA,
              "arithmetic models share the ABI's values");

namespace {

#ifndef RISE_TRACE_BLOCK
#define RISE_TRACE_BLOCK 128
#endif
constexpr int kBlock = RISE_TRACE_BLOCK;
// Waves per SIMD the traversal kernels' registers are budgeted for (96 each).
constexpr int kWaves = 5;

__device__ inline void load_ray(const float* __restrict__ rays, int64_t n, int64_t i, float& ox, float& oy, float& oz,
                                float& dx, float& dy, float& dz)
{
    ox = rays[i];
    oy = rays[n + i];
    oz = rays[2 * n + i];
    dx = rays[3 * n + i];
    dy = rays[4 * n + i];
    dz = rays[5 * n + i];
}

template <int A>
__device__ inline void init_ray_at(RayStateT<A>& r, const float* __restrict__ rays, int64_t n, int64_t i)
{
    float ox, oy, oz, dx, dy, dz;
    load_ray(rays, n, i, ox, oy, oz, dx, dy, dz);
    init_ray(r, ox, oy, oz, dx, dy, dz);
}

template <bool COUNT>
__device__ inline void flush_counts(unsigned long long* counters, unsigned nn, unsigned nt)
{
    if (COUNT) {
        atomicAdd(counters, (unsigned long long)nn);
        atomicAdd(counters + 1, (unsigned long long)nt);
    }
}

// STACK (below): node-group entries per lane held in LDS; 0 selects a private array.

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// F64: certify on the leaf records' double vertices (tri64).
template <bool COUNT, int STACK, int A, bool F64 = false>
__global__ __launch_bounds__(kBlock, kWaves) void closest_persistent(const NodeSlot* __restrict__ nodes,
                                                             const Tri48* __restrict__ tris,
                                                             const float* __restrict__ rays, int64_t n,
                                                             int32_t* __restrict__ prim_id,
                                                             float* __restrict__ t_out, unsigned long long* counters,
                                                             unsigned long long* next,
                                                             const double* __restrict__ tri64)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kBlock : 1];
    auto st = make_stack<STACK>(lds, kBlock);
    const NodeSlot* const np = nodes;
    const Tri48* const tp = tris;
    unsigned nn = 0, nt = 0;
    persist_closest<COUNT, false, F64, RayStateT<A>>(
        st, next ? grid_items(next, n) : sparse_items(n), nn, nt, np, tp, tri64,
        [&](int64_t i, RayStateT<A>& r, ClosestState& s) {
            init_ray_at(r, rays, n, i);
            closest_begin(r, s);
            return true;
        },
        [&](int64_t i, const RayStateT<A>& r, const ClosestState& s) {
            prim_id[i] = s.best_id;
            t_out[i] = s.best_id >= 0 ? (float)world_range(r, s.best_t) : INFINITY;
        });
    flush_counts<COUNT>(counters, nn, nt);
}

template <bool COUNT, int STACK, int A, bool F64 = false>
__global__ __launch_bounds__(kBlock, kWaves) void any_persistent(const NodeSlot* __restrict__ nodes,
                                                         const Tri48* __restrict__ tris,
                                                         const float* __restrict__ rays,
                                                         const float* __restrict__ tmax, int64_t n,
                                                         uint8_t* __restrict__ occluded, unsigned long long* counters,
                                                         unsigned long long* next,
                                                         const double* __restrict__ tri64)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kBlock : 1];
    auto st = make_stack<STACK>(lds, kBlock);
    const NodeSlot* const np = nodes;
    const Tri48* const tp = tris;
    unsigned nn = 0, nt = 0;
    persist_any<COUNT, false, F64, RayStateT<A>>(
        st, next ? grid_items(next, n) : sparse_items(n), nn, nt, np, tp, tri64,
        [&](int64_t i, RayStateT<A>& r, AnyState& s) {
            init_ray_at(r, rays, n, i);
            any_begin(r, scale_how_far(r, tmax ? (double)tmax[i] : kRiseInfinity), s);
            return true;
        },
        [&](int64_t i, const AnyState& s) { occluded[i] = s.hit ? 1 : 0; });
    flush_counts<COUNT>(counters, nn, nt);
}

// The closest_ex query's result staged in its rise_hip_hit slot until
// ex_records turns it into the record (keeps the record's double arithmetic
// out of the traversal loop's registers).
struct StagedHit {
    int32_t id;
    unsigned leaf;
    double t;
};
static_assert(sizeof(StagedHit) <= sizeof(rise_hip_hit), "a staged hit must fit in a hit record's slot");

// The intersection record of each ray from its staged hit, in place: the
// ray state is rebuilt from the ray as the traversal built it.
template <int A, bool F64>
__global__ __launch_bounds__(kBlock) void ex_records(const Tri48* __restrict__ tris, const float* __restrict__ rays,
                                                     int64_t n, rise_hip_hit* __restrict__ hits,
                                                     const double* __restrict__ tri64,
                                                     const double* __restrict__ attr)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const StagedHit sh = *reinterpret_cast<const StagedHit*>(hits + i);
    RayStateT<A> r;
    init_ray_at(r, rays, n, i);
    rise_hip_hit h;
    h.prim_id = sh.id;
    if (sh.id >= 0) {
        const Tri48* tri = tris + sh.leaf;
        double ab[2], nrm[3], pt[3], sn[3], uv[2];
        hit_attributes(r, tri, sh.t, ab, nrm, pt, F64 ? tri64 + 9 * (size_t)sh.leaf : nullptr,
                       attr ? attr + kAttrDoubles * (size_t)sh.leaf : nullptr, sn, uv);
        h.mesh = float_to_bits(tri->v1[3]);
        h.range = world_range(r, sh.t);
        h.alpha = ab[0];
        h.beta = ab[1];
        for (int k = 0; k < 3; ++k) {
            h.point[k] = (float)pt[k];
            h.geom_normal[k] = (float)nrm[k];
            h.shading_normal[k] = (float)sn[k];
        }
        h.uv[0] = (float)uv[0];
        h.uv[1] = (float)uv[1];
    } else {
        h.mesh = -1;
        h.range = INFINITY;
        h.alpha = h.beta = 0.0;
        for (int k = 0; k < 3; ++k) h.point[k] = h.geom_normal[k] = h.shading_normal[k] = 0.0f;
        h.uv[0] = h.uv[1] = 0.0f;
    }
    hits[i] = h;
}

// Closest hit with the face selection of rise_hip_intersect_closest_ex; the
// result is staged in hits for ex_records.
template <int STACK, int A, bool F64 = false>
__global__ __launch_bounds__(kBlock, kWaves) void closest_ex_persistent(const NodeSlot* __restrict__ nodes,
                                                                const Tri48* __restrict__ tris,
                                                                const float* __restrict__ rays, int64_t n,
                                                                unsigned faces, rise_hip_hit* __restrict__ hits,
                                                                unsigned long long* next,
                                                                const double* __restrict__ tri64,
                                                                const double* __restrict__ attr)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kBlock : 1];
    auto st = make_stack<STACK>(lds, kBlock);
    const NodeSlot* const np = nodes;
    const Tri48* const tp = tris;
    unsigned nn = 0, nt = 0;
    persist_closest<false, true, F64, RayStateT<A>>(
        st, next ? grid_items(next, n) : sparse_items(n), nn, nt, np, tp, tri64,
        [&](int64_t i, RayStateT<A>& r, ClosestState& s) {
            init_ray_at(r, rays, n, i);
            closest_begin(r, s);
            s.faces = faces;
            return true;
        },
        [&](int64_t i, const RayStateT<A>&, const ClosestState& s) {
            *reinterpret_cast<StagedHit*>(hits + i) = StagedHit{s.best_id, s.best_leaf, s.best_t};
        });
}

// Any hit with the face selection of rise_hip_intersect_any_ex.
template <int STACK, int A, bool F64 = false>
__global__ __launch_bounds__(kBlock, kWaves) void any_ex_persistent(const NodeSlot* __restrict__ nodes,
                                                            const Tri48* __restrict__ tris,
                                                            const float* __restrict__ rays,
                                                            const float* __restrict__ tmax, int64_t n,
                                                            unsigned faces, uint8_t* __restrict__ occluded,
                                                            unsigned long long* next,
                                                            const double* __restrict__ tri64)
{
    __shared__ uint2 lds[STACK > 0 ? STACK * kBlock : 1];
    auto st = make_stack<STACK>(lds, kBlock);
    const NodeSlot* const np = nodes;
    const Tri48* const tp = tris;
    unsigned nn = 0, nt = 0;
    persist_any<false, true, F64, RayStateT<A>>(
        st, next ? grid_items(next, n) : sparse_items(n), nn, nt, np, tp, tri64,
        [&](int64_t i, RayStateT<A>& r, AnyState& s) {
            init_ray_at(r, rays, n, i);
            any_begin(r, scale_how_far(r, tmax ? (double)tmax[i] : kRiseInfinity), s);
            s.faces = faces;
            return true;
        },
        [&](int64_t i, const AnyState& s) { occluded[i] = s.hit ? 1 : 0; });
}

__global__ void reset_counter(unsigned long long* c) { *c = 0ull; }

// Workgroups of a persistent launch over n rays: those resident at once (CUs x
// blocks per CU), or, when that leaves every ray kCoopLanes lanes, one wave for
// each kCoopRays rays (`sparse`; such a launch needs no fetch counter).  The
// line lies where the lanes run out: closest hits of 1000 / 7072 / 30,000 /
// 40,960 rays into 20,000 triangles take 39 / 47 / 54 / 65 us sparse, 57 / 63 / 64
// / 69 with one ray a lane from the start; into a million 131 / 171 / 228 / 244
// and 187 / 217 / 240 / 250.
struct TraceGrid {
    unsigned blocks;
    bool sparse;
};

// The cleared fetch counter of a launch, NULL for a sparse one.
unsigned long long* fetch_counter(const TraceScene& s, const TraceGrid& g, hipStream_t stream)
{
    if (g.sparse) return nullptr;
    hipLaunchKernelGGL(reset_counter, dim3(1), dim3(1), 0, stream, s.fetch_counter);
    return s.fetch_counter;
}

template <class K>
TraceGrid trace_grid(K kernel, int64_t n, bool may_be_sparse)
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess || per_cu <= 0)
        per_cu = 4;
    const int64_t want = (int64_t)cus * per_cu;
    const int64_t sparse = (n + kBlock / kCoopLanes - 1) / (kBlock / kCoopLanes);
    if (may_be_sparse && sparse <= want) return TraceGrid{(unsigned)std::max<int64_t>(1, sparse), true};
    return TraceGrid{(unsigned)std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)grid_for(n))), false};
}

}  // namespace

// The node-group stack holds at most one entry per level below the root, so
// the smallest LDS stack that fits the tree keeps occupancy highest (LDS is
// what limits waves per SIMD here).
hipError_t launch_closest(const TraceScene& s, const float* rays, int64_t n, int32_t* prim_id, float* t,
                          unsigned long long* counters, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int need = s.depth - 1;
    const dim3 block(kBlock);
#define RISE_LAUNCH_CLOSEST_F(C, S, A, F)                                                              \
    do {                                                                                               \
        const TraceGrid g = trace_grid(closest_persistent<C, S, A, F>, n, !C && S > 0);                 \
        unsigned long long* const next = fetch_counter(s, g, stream);                                  \
        hipLaunchKernelGGL((closest_persistent<C, S, A, F>), dim3(g.blocks), block, 0, stream, s.nodes, \
                           s.tris, rays, n, prim_id, t, counters, next, s.tri64);                       \
    } while (0)
#define RISE_LAUNCH_CLOSEST(C, S, A)                   \
    do {                                               \
        if (s.tri64) RISE_LAUNCH_CLOSEST_F(C, S, A, true); \
        else RISE_LAUNCH_CLOSEST_F(C, S, A, false);     \
    } while (0)
#define RISE_LAUNCH_CLOSEST_A(C, S)                                             \
    do {                                                                         \
        if (s.arith == kArithX86Fma) RISE_LAUNCH_CLOSEST(C, S, kArithX86Fma);    \
        else RISE_LAUNCH_CLOSEST(C, S, kArithIeee);                              \
    } while (0)
    if (counters) {
        if (need <= 8) RISE_LAUNCH_CLOSEST_A(true, 8);
        else if (need <= 16) RISE_LAUNCH_CLOSEST_A(true, 16);
        else RISE_LAUNCH_CLOSEST_A(true, 0);
    } else {
        if (need <= 8) RISE_LAUNCH_CLOSEST_A(false, 8);
        else if (need <= 16) RISE_LAUNCH_CLOSEST_A(false, 16);
        else RISE_LAUNCH_CLOSEST_A(false, 0);
    }
#undef RISE_LAUNCH_CLOSEST_A
#undef RISE_LAUNCH_CLOSEST
#undef RISE_LAUNCH_CLOSEST_F
    return hipGetLastError();
}

hipError_t launch_any(const TraceScene& s, const float* rays, const float* tmax, int64_t n, uint8_t* occluded,
                      unsigned long long* counters, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int need = s.depth - 1;
    const dim3 block(kBlock);
#define RISE_LAUNCH_ANY_F(C, S, A, F)                                                                   \
    do {                                                                                               \
        const TraceGrid g = trace_grid(any_persistent<C, S, A, F>, n, !C && S > 0);                     \
        unsigned long long* const next = fetch_counter(s, g, stream);                                  \
        hipLaunchKernelGGL((any_persistent<C, S, A, F>), dim3(g.blocks), block, 0, stream, s.nodes, s.tris, rays, \
                           tmax, n, occluded, counters, next, s.tri64);                                 \
    } while (0)
#define RISE_LAUNCH_ANY(C, S, A)                   \
    do {                                           \
        if (s.tri64) RISE_LAUNCH_ANY_F(C, S, A, true); \
        else RISE_LAUNCH_ANY_F(C, S, A, false);     \
    } while (0)
#define RISE_LAUNCH_ANY_A(C, S)                                             \
    do {                                                                     \
        if (s.arith == kArithX86Fma) RISE_LAUNCH_ANY(C, S, kArithX86Fma);    \
        else RISE_LAUNCH_ANY(C, S, kArithIeee);                              \
    } while (0)
    if (counters) {
        if (need <= 8) RISE_LAUNCH_ANY_A(true, 8);
        else if (need <= 16) RISE_LAUNCH_ANY_A(true, 16);
        else RISE_LAUNCH_ANY_A(true, 0);
    } else {
        if (need <= 8) RISE_LAUNCH_ANY_A(false, 8);
        else if (need <= 16) RISE_LAUNCH_ANY_A(false, 16);
        else RISE_LAUNCH_ANY_A(false, 0);
    }
#undef RISE_LAUNCH_ANY_A
#undef RISE_LAUNCH_ANY
#undef RISE_LAUNCH_ANY_F
    return hipGetLastError();
}

hipError_t launch_closest_ex(const TraceScene& s, const float* rays, int64_t n, unsigned faces, rise_hip_hit* hits,
                             hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int need = s.depth - 1;
    const dim3 block(kBlock);
#define RISE_LAUNCH_EX_F(S, A, F)                                                                           \
    do {                                                                                                    \
        const TraceGrid g = trace_grid(closest_ex_persistent<S, A, F>, n, S > 0);                           \
        unsigned long long* const next = fetch_counter(s, g, stream);                                       \
        hipLaunchKernelGGL((closest_ex_persistent<S, A, F>), dim3(g.blocks), block, 0, stream, s.nodes,     \
                           s.tris, rays, n, faces, hits, next, s.tri64, s.attr);                            \
        hipLaunchKernelGGL((ex_records<A, F>), dim3(grid_for(n)), block, 0, stream, s.tris, rays, n, hits,  \
                           s.tri64, s.attr);                                                                \
    } while (0)
#define RISE_LAUNCH_EX(S, A)                   \
    do {                                       \
        if (s.tri64) RISE_LAUNCH_EX_F(S, A, true); \
        else RISE_LAUNCH_EX_F(S, A, false);     \
    } while (0)
#define RISE_LAUNCH_EX_A(S)                                          \
    do {                                                             \
        if (s.arith == kArithX86Fma) RISE_LAUNCH_EX(S, kArithX86Fma); \
        else RISE_LAUNCH_EX(S, kArithIeee);                          \
    } while (0)
    if (need <= 8) RISE_LAUNCH_EX_A(8);
    else if (need <= 16) RISE_LAUNCH_EX_A(16);
    else RISE_LAUNCH_EX_A(0);
#undef RISE_LAUNCH_EX_A
#undef RISE_LAUNCH_EX
#undef RISE_LAUNCH_EX_F
    return hipGetLastError();
}

hipError_t launch_any_ex(const TraceScene& s, const float* rays, const float* tmax, int64_t n, unsigned faces,
                         uint8_t* occluded, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int need = s.depth - 1;
    const dim3 block(kBlock);
#define RISE_LAUNCH_EX_F(S, A, F)                                                                         \
    do {                                                                                                 \
        const TraceGrid g = trace_grid(any_ex_persistent<S, A, F>, n, S > 0);                             \
        unsigned long long* const next = fetch_counter(s, g, stream);                                    \
        hipLaunchKernelGGL((any_ex_persistent<S, A, F>), dim3(g.blocks), block, 0, stream, s.nodes, s.tris, rays, \
                           tmax, n, faces, occluded, next, s.tri64);                                      \
    } while (0)
#define RISE_LAUNCH_EX(S, A)                   \
    do {                                       \
        if (s.tri64) RISE_LAUNCH_EX_F(S, A, true); \
        else RISE_LAUNCH_EX_F(S, A, false);     \
    } while (0)
#define RISE_LAUNCH_EX_A(S)                                          \
    do {                                                             \
        if (s.arith == kArithX86Fma) RISE_LAUNCH_EX(S, kArithX86Fma); \
        else RISE_LAUNCH_EX(S, kArithIeee);                          \
    } while (0)
    if (need <= 8) RISE_LAUNCH_EX_A(8);
    else if (need <= 16) RISE_LAUNCH_EX_A(16);
    else RISE_LAUNCH_EX_A(0);
#undef RISE_LAUNCH_EX_A
#undef RISE_LAUNCH_EX
#undef RISE_LAUNCH_EX_F
    return hipGetLastError();
}

// Scratch of the allocation-free closest-hit query
// (rise_hip_intersect_closest_noalloc): word 0 is the persistent kernel's
// ray-fetch counter, cleared by a kernel at the start of every call.  A fixed
// 256 bytes per device whatever the ray count, held until the process ends.
// Host code never passes `scratch` itself to a kernel: it is a host-side
// stand-in; noalloc_scratch() returns the device's own address.
constexpr int kScratchWords = 32;
static __device__ __align__(256) unsigned long long scratch[kScratchWords];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
unsigned long long* g_scratch_ptr[kMaxScratchDevices] = {};
}  // namespace

hipError_t noalloc_scratch(unsigned long long** out)
{
    *out = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[dev] = static_cast<unsigned long long*>(p);
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

}  // namespace rise_hip
