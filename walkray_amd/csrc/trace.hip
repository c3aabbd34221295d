// trace.hip -- batch closest-hit and inside-object kernels (gfx950).
//
//  k_closest_hit        KDTree::intersect without Condition (kdtree.cpp:349-353),
//                       as used by Scene::intersect for camera rays (camera.cpp:52)
//                       and, as its NOSELF instance, with NoSelfCondition
//                       (mcRenderer.cpp:42-44, noself.cpp:13-20)
//  k_inside_object      Scene::findInsideObject (scene.cpp:115-144)
//
// One lane per ray, wave64, 256-lane workgroups; per-lane node stack in LDS;
// the finishing kernel's workgroup ids are remapped so each XCD walks a
// contiguous range of rays (neighbouring rays share chain records, and each
// XCD has its own L2).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "trace_dev.h"
#include "walk_dev.h"
#include "wr_kernels.h"

#pragma clang fp contract(off)

namespace wrd {

__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t G) {
    const uint32_t xcd = b & 7u, local = b >> 3;
    const uint32_t per = G >> 3, rem = G & 7u;
    return xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
}

// Gram-system barycentrics of Mesh::getWorldNormal (mesh.h:67-72) at o + d t.
__device__ __forceinline__ void bary(const wr_tri& T, const f3& o, const f3& d, float t, float& u1, float& u2) {
    const f3 v0 = mk(T.v0[0], T.v0[1], T.v0[2]);
    const f3 b1 = sub(mk(T.v1[0], T.v1[1], T.v1[2]), v0);
    const f3 b2 = sub(mk(T.v2[0], T.v2[1], T.v2[2]), v0);
    const f3 v = sub(add(o, muls(d, t)), v0);
    const float d12 = dot(b1, b2);
    const float l1 = len(b1);
    const float l2 = len(b2);
    const float vb1 = dot(v, b1), vb2 = dot(v, b2);
    u2 = (vb1 * d12 - vb2 * l1 * l1) / (d12 * d12 - l1 * l1 * l2 * l2);
    u1 = (vb1 - u2 * d12) / (l1 * l1);
}

__device__ __forceinline__ void add_counters(unsigned long long* out, const Counters& c) {
    unsigned long long a = c.nodes, b = c.tris, f = c.fallback;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
        f += __shfl_xor(f, off);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(out + 0, a);
        atomicAdd(out + 1, b);
        atomicAdd(out + 2, f);
    }
}

// One ray of a batch: closest-hit rays are 6 floats (origin, direction), NoSelf
// rays 8 words (origin, direction, inside, contact).
template <bool NOSELF>
__device__ __forceinline__ void load_ray(const uint32_t* __restrict__ rays, uint64_t i, f3& o, f3& d, uint32_t& inside,
                                         uint32_t& contact) {
    const uint32_t* rp = rays + (NOSELF ? 8 : 6) * i;
    o = mk(__uint_as_float(rp[0]), __uint_as_float(rp[1]), __uint_as_float(rp[2]));
    d = mk(__uint_as_float(rp[3]), __uint_as_float(rp[4]), __uint_as_float(rp[5]));
    inside = NOSELF ? rp[6] : WR_NONE;
    contact = NOSELF ? rp[7] : WR_NONE;
}

template <bool NOSELF>
__device__ __forceinline__ NoSelf make_noself(const SceneDev& S, const wr_tree_hdr& H, uint32_t inside,
                                              uint32_t contact) {
    if (!NOSELF) return NoSelf{};
    return NoSelf{inside, contact, S.rec_nrm + 9 * (size_t)H.rec_base, S.obj_has_normals};
}

// Fast pass of the batch closest-hit query as a persistent kernel, for batches
// of more rays than the device holds lanes: a wave takes one unit of 64 rays
// at a time and refills a lane with the next ray as soon as its traversal
// ends, so a wave never waits for its slowest ray.  The result of the fast
// pass (record, t, first record of the leaf, overflow flag) goes to hits[ray];
// k_closest_hit_finish completes it.
// The units come from a UnitQueue.  With one counter atomic per wave and 256
// rays, probing of the other seven ranges at the end and a count of finished
// waves, 400,009 incoherent rays on the 512-object field took 242 us and 8M
// camera rays 0.93 ms; now 142 us and 0.80 ms (with the finishing kernel;
// 16.8M rays on the 2.1M-triangle heightfield, where the traversal itself is
// all, stay at 2.6 ms coherent, 3.2 ms incoherent).
// Compiled for 8 waves per SIMD (64 VGPRs): more waves in flight hide more of
// the node-fetch latency; with the NoSelf test for the 5 that its registers
// allow.
// Scheduling knobs (ChTune, chosen by the autotuner): idle lanes are refilled
// once at least refill_min are idle; a wave runs node-only steps while at
// least node_phase_min lanes sit at wide nodes (a mixed step pays for both the
// node code and the triangle code).
// D: stack levels in LDS (the autotuner's stack-depth knob).
template <bool NOSELF, bool COUNT, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NOSELF ? 5 : 8))) void k_closest_hit(
    SceneDev S, wr_tree_hdr H, const uint32_t* __restrict__ rays, uint64_t n, uint4* __restrict__ hits,
    unsigned long long* counters, unsigned long long* work, uint32_t refill_min, uint32_t node_phase_min,
    uint32_t batch, uint32_t first, uint32_t stripe) {
    const Tree tr = make_tree(H, S);
    StackSpillT<D> spill;
    LaneStackT<D> st(&spill);
    Counters cnt{0, 0, 0};
    NoSelf ns{};
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    __shared__ unsigned long long pool;
    UnitQueue queue;
    queue.init(&pool, work, (uint32_t)((n + 63) / 64), gridDim.x, first, batch, stripe);
    uint64_t bnext = 0, bend = 0;  // the rays of the wave's current unit [bnext, bend)
    bool exhausted = false;
    bool active = false, overflow = false;
    uint64_t rid = 0;
    uint32_t ref = 0;
    RayPre r{};
    HitState h{};
    for (;;) {
        uint64_t idle = __ballot(!active);
        if (!exhausted && (uint32_t)__popcll(idle) >= refill_min) {
            while (idle != 0) {
                if (bnext == bend) {
                    const uint32_t u = queue.next();
                    if (u == WR_NONE) {
                        exhausted = true;
                        break;
                    }
                    bnext = 64ull * u;
                    bend = bnext + 64 < n ? bnext + 64 : n;
                }
                const uint64_t avail = bend - bnext;
                const uint64_t rank = (uint64_t)__popcll(idle & below);
                if (!active && rank < avail) {
                    rid = bnext + rank;
                    f3 o, d;
                    uint32_t inside, contact;
                    load_ray<NOSELF>(rays, rid, o, d, inside, contact);
                    r = make_ray(o, d, tr.scale);
                    ns = make_noself<NOSELF>(S, H, inside, contact);
                    overflow = false;
                    if (wide_begin(tr, r, st, h, ref)) active = true;
                    else hits[rid] = make_uint4(WR_NONE, 0u, 0u, 0u);  // misses the root box
                }
                const uint64_t took = (uint64_t)__popcll(idle);
                bnext += took < avail ? took : avail;
                idle = __ballot(!active);
            }
        }
        if (__ballot(active) == 0) break;  // only once the counter is exhausted
        // node phase: while at least node_phase_min lanes sit at wide nodes, only
        // those lanes step (no triangle code runs); then one step for every lane
        for (;;) {
            const bool at_node = active && !(ref & WR_LEAF_BIT);
            if ((uint32_t)__popcll(__ballot(at_node)) < node_phase_min) break;
            if (at_node && !wide_step<NOSELF, COUNT>(tr, r, ns, st, h, ref, overflow, cnt)) {
                hits[rid] = make_uint4(h.rec, __float_as_uint(h.t), h.leaf, overflow ? 1u : 0u);
                active = false;
            }
        }
        if (active && !wide_step<NOSELF, COUNT>(tr, r, ns, st, h, ref, overflow, cnt)) {
            hits[rid] = make_uint4(h.rec, __float_as_uint(h.t), h.leaf, overflow ? 1u : 0u);
            active = false;
        }
    }
    if (COUNT) add_counters(counters, cnt);
}

// Completion of one ray's fast pass (binary fast pass after a wide-stack
// overflow, chain verification, exact fallback) and its output record.
template <bool NOSELF, bool COUNT, class Stack>
__device__ __forceinline__ uint4 complete_hit(const Tree& tr, const RayPre& r, const NoSelf& ns, Stack& st,
                                              Counters& cnt, HitState h, bool overflow) {
    uint4 out = make_uint4(WR_NONE, __float_as_uint(-1.f), 0u, 0u);
    bool failed;
    // the winner's record is fetched alongside the verification's first fetch
    const uint32_t rec0 = h.rec;
    wr_tri T{};
    if (rec0 != WR_NONE) T = tr.tris[rec0];
    finish_hit<NOSELF, COUNT>(tr, r, ns, st, cnt, h, overflow, failed);
    if (h.rec != WR_NONE) {
        if (h.rec != rec0) T = tr.tris[h.rec];
        float u1, u2;
        bary(T, r.o, r.d, h.t, u1, u2);
        out = make_uint4(T.prim, __float_as_uint(h.t), __float_as_uint(u1), __float_as_uint(u2));
    }
    if (failed) out.x = 0xFFFFFFFEu;  // stack overflow: reported, never silently wrong
    return out;
}

// Completion of k_closest_hit's records, one lane per ray, so the verification
// walks of a wave run together.
template <bool NOSELF, bool COUNT, int D>
__global__ __launch_bounds__(256) void k_closest_hit_finish(SceneDev S, wr_tree_hdr H,
                                                            const uint32_t* __restrict__ rays, uint64_t n,
                                                            uint4* __restrict__ hits, unsigned long long* counters,
                                                            unsigned long long* work) {
    if (blockIdx.x == 0) UnitQueue::clear(work);  // for the next launch
    const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
    const uint64_t i = (uint64_t)b * 256 + threadIdx.x;
    Counters cnt{0, 0, 0};
    StackSpillT<D> spill;
    LaneStackT<D> st(&spill);
    if (i < n) {
        const uint4 f = hits[i];
        const HitState h{__uint_as_float(f.y), f.x, f.z};
        const bool overflow = f.w != 0;
        uint4 out = make_uint4(WR_NONE, __float_as_uint(-1.f), 0u, 0u);
        if (h.rec != WR_NONE || overflow) {
            f3 o, d;
            uint32_t inside, contact;
            load_ray<NOSELF>(rays, i, o, d, inside, contact);
            const Tree tr = make_tree(H, S);
            const RayPre r = make_ray(o, d, tr.scale);
            out = complete_hit<NOSELF, COUNT>(tr, r, make_noself<NOSELF>(S, H, inside, contact), st, cnt, h, overflow);
        }
        hits[i] = out;
    }
    if (COUNT) add_counters(counters, cnt);
}

// The whole query in one launch, one lane per ray: the first `width` lanes of
// every wave take a ray each.  A small batch is bound by the latency of its
// longest traversal (about 40 us), and lanes that share a wave lengthen it:
// they wait for each other's triangle and node steps, and their 64 B fetches
// go through one CU's cache one line at a time.  So few rays are spread over
// many waves.  1,000 / 16,000 / 65,537 rays on the 512-object field: 60 / 77 /
// 80 us with 16 lanes, 46 / 106 / 207 us with one, 67 / 95 / 91 us with 64.
template <bool NOSELF>
__global__ __launch_bounds__(256) void k_closest_hit_small(SceneDev S, wr_tree_hdr H,
                                                           const uint32_t* __restrict__ rays, uint64_t n,
                                                           uint32_t width, bool by_xcd, uint4* __restrict__ hits) {
    const uint32_t block = by_xcd ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const uint32_t lane = threadIdx.x & 63u, wave = block * 4 + (threadIdx.x >> 6);
    const uint64_t i = (uint64_t)wave * width + lane;
    if (lane >= width || i >= n) return;
    StackSpill spill;
    LaneStack st(&spill);
    f3 o, d;
    uint32_t inside, contact;
    load_ray<NOSELF>(rays, i, o, d, inside, contact);
    const Tree tr = make_tree(H, S);
    const RayPre r = make_ray(o, d, tr.scale);
    const NoSelf ns = make_noself<NOSELF>(S, H, inside, contact);
    Counters cnt{0, 0, 0};
    HitState h;
    bool overflow;
    traverse_wide<NOSELF, false>(tr, r, ns, st, h, overflow, cnt);
    hits[i] = complete_hit<NOSELF, false>(tr, r, ns, st, cnt, h, overflow);
}

// The fast pass of a path walk's step (walk_dev.h): the *n_dev rays, NoSelf,
// spread over the chip as k_wf_trace spreads its paths: a unit of up to 64 rays
// for each of kSpread waves, and no more lanes of a wave at work than that.
__global__ __launch_bounds__(256) void k_walk_trace(SceneDev S, wr_tree_hdr H, const uint32_t* __restrict__ rays,
                                                    const uint32_t* n_dev, uint4* __restrict__ hits,
                                                    unsigned long long* work) {
    constexpr uint32_t kSpread = 4096, kRefillMin = 16, kNodePhaseMin = 32;
    const uint32_t n = *n_dev;
    if (n <= wr::kWalkFew) return;  // k_walk_shade traces the last paths itself
    uint32_t width = 1;
    while (width < 64 && 2ull * n > 3ull * width * kSpread) width *= 2;
    const uint32_t units = (uint32_t)(((uint64_t)n + width - 1) / width);
    const uint32_t used = min((units + 31) / 32 * 8, gridDim.x);
    if (blockIdx.x >= used) return;
    const Tree tr = make_tree(H, S);
    StackSpill spill;
    LaneStack st(&spill);
    Counters cnt{0, 0, 0};
    NoSelf ns{};
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t lanes = width < 64 ? (1ull << width) - 1ull : ~0ull;  // the lanes that take rays
    const uint32_t refill_min = width < 64 ? 1u : kRefillMin;
    const uint32_t node_phase_min = (width * kNodePhaseMin + 63) / 64;
    __shared__ unsigned long long pool;
    UnitQueue queue;
    queue.init(&pool, work, units, used, 4, units / used > 12 ? 2 : 1,
               units > 4 * used ? min(max(units / (16 * wr::kXcds), 1u), 64u) : 1u);
    uint32_t bnext = 0, bend = 0;  // the rays of the wave's current unit [bnext, bend)
    bool exhausted = false;
    bool active = false, overflow = false;
    uint32_t rid = 0, ref = 0;
    RayPre r{};
    HitState h{};
    for (;;) {
        uint64_t idle = __ballot(!active) & lanes;
        if (!exhausted && (uint32_t)__popcll(idle) >= refill_min) {
            while (idle != 0) {
                if (bnext == bend) {
                    const uint32_t u = queue.next();
                    if (u == WR_NONE) {
                        exhausted = true;
                        break;
                    }
                    bnext = u * width;
                    bend = n - bnext > width ? bnext + width : n;
                }
                const uint32_t avail = bend - bnext;
                const uint32_t rank = (uint32_t)__popcll(idle & below);
                if (!active && lane < width && rank < avail) {
                    rid = bnext + rank;
                    f3 o, d;
                    uint32_t inside, contact;
                    load_ray<true>(rays, rid, o, d, inside, contact);
                    r = make_ray(o, d, tr.scale);
                    ns = make_noself<true>(S, H, inside, contact);
                    overflow = false;
                    if (wide_begin(tr, r, st, h, ref)) active = true;
                    else hits[rid] = make_uint4(WR_NONE, 0u, 0u, 0u);  // misses the root box
                }
                const uint32_t took = (uint32_t)__popcll(idle);
                bnext += took < avail ? took : avail;
                idle = __ballot(!active) & lanes;
            }
        }
        if (__ballot(active) == 0) break;  // only once the queue is empty
        for (;;) {
            const bool at_node = active && !(ref & WR_LEAF_BIT);
            if ((uint32_t)__popcll(__ballot(at_node)) < node_phase_min) break;
            if (at_node && !wide_step<true, false>(tr, r, ns, st, h, ref, overflow, cnt)) {
                hits[rid] = make_uint4(h.rec, __float_as_uint(h.t), h.leaf, overflow ? 1u : 0u);
                active = false;
            }
        }
        if (active && !wide_step<true, false>(tr, r, ns, st, h, ref, overflow, cnt)) {
            hits[rid] = make_uint4(h.rec, __float_as_uint(h.t), h.leaf, overflow ? 1u : 0u);
            active = false;
        }
    }
}

__global__ __launch_bounds__(256) void k_inside_object(SceneDev S, const uint32_t* __restrict__ rays, uint64_t n,
                                                       uint32_t* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    StackSpill spill;
    LaneStack st(&spill);
    const uint32_t* rp = rays + 8 * i;
    const f3 o = mk(__uint_as_float(rp[0]), __uint_as_float(rp[1]), __uint_as_float(rp[2]));
    const f3 d = mk(__uint_as_float(rp[3]), __uint_as_float(rp[4]), __uint_as_float(rp[5]));
    out[i] = find_inside(S, o, d, rp[7], st);
}

// Global triangle id -> (object, triangle of the object) for a batch of hits
// (ObjSourceInfo, scene.cpp:34-36,110): the last object whose first global
// triangle is <= prim, found by binary search over the object table.
__global__ __launch_bounds__(256) void k_hit_sources(const wr_object_gpu* __restrict__ objs, uint32_t n_objs,
                                                     uint32_t n_tris, const uint4* __restrict__ hits, uint64_t n,
                                                     uint32_t* __restrict__ obj, uint32_t* __restrict__ tri) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t prim = hits[i].x;
    uint32_t o = WR_NONE, t = WR_NONE;
    if (prim < n_tris) {
        uint32_t lo = 0, hi = n_objs;  // first object with prim_base > prim lies in [lo, hi]
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (objs[mid].prim_base <= prim) lo = mid + 1;
            else hi = mid;
        }
        o = lo - 1;
        t = prim - objs[o].prim_base;
    }
    obj[i] = o;
    tri[i] = t;
}

}  // namespace wrd

namespace wr {

hipError_t launch_hit_sources(const SceneDev& S, uint32_t n_tris, const void* hits, uint64_t n, uint32_t* obj,
                              uint32_t* tri, hipStream_t st) {
    if (n == 0) return hipSuccess;
    wrd::k_hit_sources<<<(uint32_t)((n + 255) / 256), 256, 0, st>>>(S.objs, S.n_objs, n_tris, (const uint4*)hits, n,
                                                                     obj, tri);
    return hipGetLastError();
}

// Workgroups of the persistent kernel with D LDS stack levels: per_cu per CU
// (0: as many as fit).
template <bool NOSELF, int D>
static uint32_t persistent_blocks(uint64_t n, uint32_t per_cu_want) {
    static int cus = 0, per_cu_max = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu_max, wrd::k_closest_hit<NOSELF, false, D>, 256,
                                                         wrd::stack_lds_bytes<D>()) != hipSuccess ||
            cus <= 0 || per_cu_max <= 0) {
            cus = 256;
            per_cu_max = 1;
        }
    }
    const uint32_t per_cu = per_cu_want && per_cu_want < (uint32_t)per_cu_max ? per_cu_want : (uint32_t)per_cu_max;
    const uint64_t resident = (uint64_t)cus * per_cu;
    const uint64_t need = (n + 255) / 256;
    return (uint32_t)(need < resident ? need : resident);
}

// Waves that k_closest_hit_small spreads a small batch over: four per SIMD.
constexpr uint64_t kSmallWaves = 4096;
// Largest batch for k_closest_hit_small; a larger one has more rays than the
// persistent kernel's resident lanes (8 waves on each of 1,024 SIMDs), so that
// refilling lanes pays.  Incoherent rays on the field, in us, small against
// persistent: 400,009 rays 132 / 142, 700,001 rays 178 / 181, 1,000,003 rays
// 229 / 207, 4M 762 / 459.  With the NoSelf test, whose normals leave both
// kernels 5 waves per SIMD, rays from camera hits cross over later: 1M
// 181 / 255, 2M 306 / 367, 4M 564 / 555.
template <bool NOSELF>
constexpr uint64_t kSmallMax = NOSELF ? 1ull << 21 : kClosestHitOneLaunch;

// NoSelf batches continue paths: neighbouring rays start near each other, their
// normals leave the kernel 5 waves per SIMD, and in a small tree they mostly
// read what the XCD's L2 already holds.  There, between these numbers of rays,
// full waves in the order in which each XCD walks its own range are the faster:
// 100,000 rays on 16 / 40 / 64 objects 50 / 61 / 68 us so, 58 / 67 / 73 us spread
// (150,000: 55 / 65 / 74 and 65 / 74 / 83); from 200,000 rays on, or from 100
// objects (96,000 triangles) on, spreading is.
constexpr uint64_t kLocalMin = 49152, kLocalMax = 196608;
constexpr uint32_t kLocalTris = 81920;
// In a larger tree eight lanes a wave up to this number of rays (two rounds of
// the waves that fit): 50,000 rays on 512 objects 86 us, 104 with sixteen.
constexpr uint64_t kNarrowMax = 65536;

template <bool NOSELF, int D>
static hipError_t launch_closest_hit_d(const SceneDev& S, const wr_tree_hdr& H, const uint32_t* rays, uint64_t n,
                                       void* hits, unsigned long long* counters, unsigned long long* work,
                                       uint32_t per_cu, uint32_t rmin, uint32_t nmin, uint32_t batch,
                                       hipStream_t st) {
    uint4* out = (uint4*)hits;
    if (n <= kSmallMax<NOSELF> && !counters) {
        // the power of two nearest to the rays per wave
        uint32_t width = 1;
        while (width < 64 && 2 * n > 3ull * width * kSmallWaves) width *= 2;
        const bool by_xcd = NOSELF && H.n_recs <= kLocalTris && n > kLocalMin && n <= kLocalMax;
        if (by_xcd) width = 64;
        else if (NOSELF && n <= kNarrowMax) width = std::min(width, 8u);
        const uint64_t waves = (n + width - 1) / width;
        wrd::k_closest_hit_small<NOSELF>
            <<<(uint32_t)((waves + 3) / 4), 256, wrd::kStackLdsBytes, st>>>(S, H, rays, n, width, by_xcd, out);
        return hipGetLastError();
    }
    const uint32_t pgrid = persistent_blocks<NOSELF, D>(n, per_cu);
    const uint32_t grid = (uint32_t)((n + 255) / 256);
    const size_t lds = wrd::stack_lds_bytes<D>();
    // units of 64 rays: a workgroup's first ones, one for each of its waves; then at most `batch` rays
    // at a time, fewer where it would come back less than eight times; stripes of at most 64
    const uint64_t units = (n + 63) / 64;
    const uint32_t first = (uint32_t)std::min<uint64_t>((units + pgrid - 1) / pgrid, 4);
    const uint64_t left = units > (uint64_t)first * pgrid ? units - (uint64_t)first * pgrid : 0;
    const uint32_t take = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(batch / 64, left / (8ull * pgrid)));
    const uint32_t stripe = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(64, units / (16 * kXcds)));
    if (counters) {
        wrd::k_closest_hit<NOSELF, true, D>
            <<<pgrid, 256, lds, st>>>(S, H, rays, n, out, counters, work, rmin, nmin, take, first, stripe);
        wrd::k_closest_hit_finish<NOSELF, true, D><<<grid, 256, lds, st>>>(S, H, rays, n, out, counters, work);
    } else {
        wrd::k_closest_hit<NOSELF, false, D>
            <<<pgrid, 256, lds, st>>>(S, H, rays, n, out, nullptr, work, rmin, nmin, take, first, stripe);
        wrd::k_closest_hit_finish<NOSELF, false, D><<<grid, 256, lds, st>>>(S, H, rays, n, out, nullptr, work);
    }
    return hipGetLastError();
}

hipError_t launch_closest_hit(const SceneDev& S, const wr_tree_hdr& H, const float* rays_f, uint64_t n, void* hits,
                              unsigned long long* counters, unsigned long long* work, const ChTune& tune,
                              hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t* rays = (const uint32_t*)rays_f;
    // refill_min in [1, 64]; node_phase_min in [1, 65] (0 would never leave the node phase; 65 disables it)
    const uint32_t rmin = tune.refill_min < 1 ? 1 : (tune.refill_min > 64 ? 64 : tune.refill_min);
    const uint32_t nmin = tune.node_phase_min < 1 ? 1 : (tune.node_phase_min > 65 ? 65 : tune.node_phase_min);
    // rays per work-counter atomic in [64, 4096]
    const uint32_t batch = tune.batch < 64 ? 64 : (tune.batch > 4096 ? 4096 : tune.batch);
    const uint32_t pc = tune.blocks_per_cu;
    switch (tune.lds_levels) {
        case 4:
            return launch_closest_hit_d<false, 4>(S, H, rays, n, hits, counters, work, pc, rmin, nmin, batch, st);
        case 16:
            return launch_closest_hit_d<false, 16>(S, H, rays, n, hits, counters, work, pc, rmin, nmin, batch, st);
        default:
            return launch_closest_hit_d<false, 8>(S, H, rays, n, hits, counters, work, pc, rmin, nmin, batch, st);
    }
}

hipError_t launch_closest_hit_path(const SceneDev& S, const wr_tree_hdr& H, const uint32_t* rays, uint64_t n,
                                   void* hits, unsigned long long* work, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const ChTune t;
    return launch_closest_hit_d<true, 8>(S, H, rays, n, hits, nullptr, work, t.blocks_per_cu, t.refill_min,
                                         t.node_phase_min, t.batch, st);
}

hipError_t launch_walk_trace(const SceneDev& S, const wr_tree_hdr& H, const uint32_t* rays, const uint32_t* n,
                             uint32_t max_n, uint4* hits, unsigned long long* work, hipStream_t st) {
    // as many workgroups as fit (5 waves per SIMD), or as the rays can use
    static const uint32_t resident = [] {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wrd::k_walk_trace, 256, wrd::kStackLdsBytes) !=
                hipSuccess || cus <= 0 || per_cu <= 0)
            return 256u;
        return (uint32_t)(cus * per_cu);
    }();
    const uint32_t grid = (uint32_t)std::min<uint64_t>(((uint64_t)max_n + 31) / 32 * 8, resident);
    wrd::k_walk_trace<<<grid, 256, wrd::kStackLdsBytes, st>>>(S, H, rays, n, hits, work);
    return hipGetLastError();
}

hipError_t launch_inside_object(const SceneDev& S, uint32_t max_obj_depth, const uint32_t* rays, uint64_t n,
                                uint32_t* out, hipStream_t st) {
    (void)max_obj_depth;
    if (n == 0) return hipSuccess;
    const uint32_t grid = (uint32_t)((n + 255) / 256);
    wrd::k_inside_object<<<grid, 256, wrd::kStackLdsBytes, st>>>(S, rays, n, out);
    return hipGetLastError();
}

}  // namespace wr
