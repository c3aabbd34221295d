// walk_dev.h -- MCRenderer::samplePath (mcRenderer.cpp:16-57) for many paths at
// once, one ray of every path per step: the sub-paths of
// BidirectionalPathTracer and VCMTracer, light paths, and PhotonMap's eye paths.
//
// A lane that ran its whole path kept its wave for the longest of 64 paths, in
// every traversal for the longest of 64 rays, with the registers of all of
// samplePath.  Here a step traces the live paths' rays in a kernel of its own
// (k_walk_trace, lanes refilled as in the closest-hit batches) and
// k_walk_shade<P> completes the hits, scatters, and appends the paths that go
// on to the next step's list.  The work of a step is bound by its traversals
// where many paths live and by the latency of the longest one where few do, so
// the trace spreads few paths over many waves.  The paths' random numbers are
// keyed by path and vertex, so the order of a list changes no path.
// 2 x 524,288 sub-paths in the Cornell box (maxPathLen 8): 5.2 ms as one kernel,
// 2.5 ms in steps.
#pragma once
#include <hip/hip_runtime.h>

#include "pt_dev.h"
#include "wr_capi_internal.h"

#pragma clang fp contract(off)

namespace wr {
// A step with at most this many live paths ends the walk: what bounds it is the
// latency of one traversal and one vertex (about 62 us in k_walk_shade, whose
// registers spill), to which two kernels' launches and the lists add 25 us, so
// k_walk_shade takes the paths to their ends, spread over the chip.  307,200 light paths of the object field
// (maxPathLen 16) with their photons and grid 2.30 ms without, 2.0 ms up to
// 16,384 paths, 1.91 up to 32,768, 1.79 up to 65,536 and 131,072, where
// PhotonMap loses 1.5%.
constexpr uint32_t kWalkFew = 65536;
// List steps of a walk: every step of the renderers (maxPathLen up to 32).  A
// longer walk's paths that are still alive then are taken to their ends like
// the last few, so that a call's launches do not grow with its path length:
// 1,000 light paths with a limit of 1,000 scatters launched 2,000 kernels that
// found nothing to do: 5.2 ms, 0.28 now.
constexpr uint32_t kWalkListSteps = 33;
}  // namespace wr

namespace wrd {

// The live paths of two consecutive steps: rays in the batch NoSelf layout (8
// words: origin, direction, inside, contact) and the paths they belong to.
struct WalkLists {
    uint32_t* rays[2];
    uint32_t* path[2];
    uint4* hits;               // the step's fast-pass results
    uint32_t* n;               // n[s]: live paths of step s, zero where not reached
    unsigned long long* work;  // the trace's unit counters
};

__device__ __forceinline__ void put_walk_ray(const WalkLists& W, uint32_t step, uint32_t j, uint32_t path, f3 o, f3 d,
                                             uint32_t inside, uint32_t contact) {
    uint32_t* r = W.rays[step & 1] + 8 * (size_t)j;
    r[0] = __float_as_uint(o.x); r[1] = __float_as_uint(o.y); r[2] = __float_as_uint(o.z);
    r[3] = __float_as_uint(d.x); r[4] = __float_as_uint(d.y); r[5] = __float_as_uint(d.z);
    r[6] = inside;
    r[7] = contact;
    W.path[step & 1][j] = path;
}

// The first rays.  P::begin(sc, path, st, o, d, inside, contact): the path's
// first record and ray (inside and contact of its NoSelf condition), false for
// a path that ends there.
template <class P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_walk_begin(SceneDev S, P policy,
                                                                                           WalkLists W, uint32_t path0,
                                                                                           uint32_t n_paths) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, path = path0 + i;
    StackSpill spill;
    LaneStack st(&spill);
    const SceneCtx sc = make_scene_ctx(S);
    f3 o, d;
    uint32_t inside, contact;
    const bool go = i < n_paths && policy.begin(sc, path, st, o, d, inside, contact);
    const uint32_t j = block_append(W.n, go);
    if (go) put_walk_ray(W, 0, j, path, o, d, inside, contact);
}

// Step s: completes every live path's hit and takes the path one vertex on.
// P::step(sc, path, s, o, d, hit, st, out): the vertex at the hit (hit.rec
// WR_NONE: the ray escaped); true if the path goes on with out.
// LAST: the walk's last launch, which takes any number of paths to their ends.
template <class P, bool LAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_walk_shade(SceneDev S, P policy,
                                                                                           WalkLists W, uint32_t s) {
    const uint32_t n = W.n[s];
    if (blockIdx.x == 0) UnitQueue::clear(W.work);  // for the next step's trace
    StackSpill spill;
    LaneStack st(&spill);
    const SceneCtx sc = make_scene_ctx(S);
    if (LAST || n <= wr::kWalkFew) {  // the rest of every path, the trace included
        uint32_t width = 1;           // lanes of a wave that take a path
        while (width < 64 && (uint64_t)width * gridDim.x * 4 < n) width *= 2;
        const uint32_t lane = threadIdx.x & 63u;
        if (lane >= width) return;
        for (uint32_t i = (blockIdx.x * 4 + (threadIdx.x >> 6)) * width + lane; i < n;
             i = LAST ? i + gridDim.x * 4 * width : n) {
            const uint32_t path = W.path[s & 1][i];
            const uint32_t* rp = W.rays[s & 1] + 8 * (size_t)i;
            Out out;
            out.o = mk(__uint_as_float(rp[0]), __uint_as_float(rp[1]), __uint_as_float(rp[2]));
            out.d = mk(__uint_as_float(rp[3]), __uint_as_float(rp[4]), __uint_as_float(rp[5]));
            out.inside = rp[6];
            out.contact = rp[7];
            for (uint32_t k = s;; k++) {
                const f3 o = out.o, d = out.d;
                const PHit hit = trace_scene<true>(sc, o, d, out.inside, out.contact, st);
                if (!policy.step(sc, path, k, o, d, hit, st, out)) break;
            }
        }
        return;
    }
    for (uint32_t i0 = blockIdx.x * 256; i0 < n; i0 += gridDim.x * 256) {
        const uint32_t i = i0 + threadIdx.x;
        bool go = false;
        uint32_t path = 0;
        Out out;
        if (i < n) {
            path = W.path[s & 1][i];
            const uint32_t* rp = W.rays[s & 1] + 8 * (size_t)i;
            const f3 o = mk(__uint_as_float(rp[0]), __uint_as_float(rp[1]), __uint_as_float(rp[2]));
            const f3 d = mk(__uint_as_float(rp[3]), __uint_as_float(rp[4]), __uint_as_float(rp[5]));
            const uint4 f = W.hits[i];
            HitState h{__uint_as_float(f.y), f.x, f.z};
            const bool overflow = f.w != 0;
            if (h.rec != WR_NONE || overflow) {
                const RayPre r = make_ray(o, d, sc.tr.scale);
                const NoSelf ns{rp[6], rp[7], sc.gnrm, S.obj_has_normals};
                Counters cnt{0, 0, 0};
                bool failed;
                finish_hit<true, false>(sc.tr, r, ns, st, cnt, h, overflow, failed);
            }
            PHit hit;
            hit.t = h.t;
            hit.rec = h.rec;
            hit.obj = h.rec == WR_NONE ? WR_NONE : sc.tr.tris[h.rec].obj;
            go = policy.step(sc, path, s, o, d, hit, st, out);
        }
        const uint32_t j = block_append(W.n + s + 1, go);
        if (go) put_walk_ray(W, s + 1, j, path, out.o, out.d, out.inside, out.contact);
    }
}

}  // namespace wrd

namespace wr {

// The trace of a walk's step (trace.hip): the fast pass, with NoSelf, of the
// *n rays (device; at most max_n).
hipError_t launch_walk_trace(const SceneDev& S, const wr_tree_hdr& H, const uint32_t* rays, const uint32_t* n,
                             uint32_t max_n, uint4* hits, unsigned long long* work, hipStream_t st);

// Walks n_paths paths of at most `steps` rays each, enqueued on the context's
// stream.  The lists (88 B a path) are scratch, so a long call runs 4M paths
// at a time, fewer where the device has no room for them.
template <class P>
hipError_t run_walk(wr_ctx* ctx, const SceneDev& S, const wr_tree_hdr& H, const P& policy, uint32_t n_paths,
                    uint32_t steps) {
    hipStream_t st = ctx->stream;
    wrd::WalkLists W;
    W.work = ctx->d_work;
    uint32_t chunk = n_paths < (1u << 22) ? n_paths : (1u << 22);
    Scratch mem(*ctx->pool);
    char* lists = nullptr;
    hipError_t e;
    while ((e = mem.get(&lists, 88ull * chunk)) == hipErrorOutOfMemory && chunk > (1u << 14)) {
        (void)hipGetLastError();  // must not surface at a later launch check
        chunk /= 4;
    }
    if (e != hipSuccess) return e;
    const uint32_t lists_max = steps < kWalkListSteps ? steps : kWalkListSteps;
    if ((e = mem.get(&W.n, sizeof(uint32_t) * (lists_max + 1))) != hipSuccess) return e;
    for (int k = 0; k < 2; k++) W.rays[k] = (uint32_t*)(lists + 32ull * chunk * k);
    W.hits = (uint4*)(lists + 64ull * chunk);
    for (int k = 0; k < 2; k++) W.path[k] = (uint32_t*)(lists + (80ull + 4 * k) * chunk);
    for (uint32_t p = 0; p < n_paths;) {
        const uint32_t n = n_paths - p < chunk ? n_paths - p : chunk;
        const uint32_t blocks = (n + 255) / 256;
        if ((e = hipMemsetAsync(W.n, 0, sizeof(uint32_t) * (lists_max + 1), st)) != hipSuccess) return e;
        // at least one wave per SIMD for a few paths' ends
        const uint32_t shade = blocks < 256 ? 256 : (blocks < 2048 ? blocks : 2048);
        wrd::k_walk_begin<P><<<blocks, 256, wrd::kStackLdsBytes, st>>>(S, policy, W, p, n);
        const uint32_t list_steps = n <= kWalkFew ? 0 : lists_max;  // a few paths end in the first shade
        for (uint32_t s = 0; s < list_steps; s++) {
            e = launch_walk_trace(S, H, W.rays[s & 1], W.n + s, n, W.hits, W.work, st);
            if (e != hipSuccess) return e;
            wrd::k_walk_shade<P, false><<<shade, 256, wrd::kStackLdsBytes, st>>>(S, policy, W, s);
        }
        if (list_steps < steps)
            wrd::k_walk_shade<P, true><<<shade, 256, wrd::kStackLdsBytes, st>>>(S, policy, W, list_steps);
        p += n;
    }
    return hipGetLastError();
}

}  // namespace wr
