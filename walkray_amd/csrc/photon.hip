// photon.hip -- light sub-paths and the photon hash grid (gfx950), with their
// C ABI entry points.
//
//  light paths      Scene::genLightSample as AbstractObject::genSurfaceSample
//                   (abstractObj.cpp:18-52) and MCRenderer::samplePath
//                   (mcRenderer.cpp:16-57) from it as a path walk (LightWalk),
//                   every Ray of the Path written as a 64 B record.
//  photon collect   count, scan and write the light points VCM / PPM keep
//                   (vcmTracer.cpp:42-55): deterministic, path-major order.
//  hash grid        HashGrid::Build (hashgrid.hxx:24-75) as bbox reduction and
//                   a stable radix sort of (cell, point) pairs (mIndices: the
//                   serial scatter keeps input order inside a cell, so does a
//                   stable sort; mCellEnds: the cells' ends in the sorted
//                   pairs); HashGrid::Process (hashgrid.hxx:77-158) as a range
//                   query, one lane per query point.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "grid_dev.h"
#include "pt_dev.h"
#include "walk_dev.h"
#include "wr_capi_internal.h"

#pragma clang fp contract(off)

namespace wrd {

// Vertex counters of a light path's uniforms: kLightVertex (light pick and
// point), kLightVertex + 1 (direction), kLightVertex + 2 + d (scatter at depth d).
constexpr uint32_t kLightVertex = 0x80000000u;

__device__ __forceinline__ void put_vertex(wr_path_vertex& v, f3 o, f3 d, f3 rad, float op, float dp, uint32_t contact,
                                           uint32_t ctri, uint32_t inside, bool delta) {
    v.origin[0] = o.x; v.origin[1] = o.y; v.origin[2] = o.z;
    v.direction[0] = d.x; v.direction[1] = d.y; v.direction[2] = d.z;
    v.radiance[0] = rad.x; v.radiance[1] = rad.y; v.radiance[2] = rad.z;
    v.origin_prob = op;
    v.direction_prob = dp;
    v.contact_obj = contact;
    v.contact_tri = contact == WR_NONE ? 0u : ctri;
    v.inside_obj = inside;
    v.flags = delta ? (uint32_t)WR_VERTEX_DELTA : 0u;
    v.pad = 0u;
}

// terminateRay (mcRenderer.cpp:20-27): the origin of the ray passed in.
__device__ __forceinline__ void put_terminate(wr_path_vertex& v, f3 o) {
    const f3 z = mk(0.f, 0.f, 0.f);
    put_vertex(v, o, z, z, 1.f, 1.f, WR_NONE, 0u, WR_NONE, true);
}

// The light paths path0 + k, k < n, as a path walk (walk_dev.h): record s + 1 of
// path k is written by step s.  As one kernel, a lane per path, 307,200 paths
// of the object field (maxPathLen 16) took 2.0 ms; in steps 1.5 ms.
struct LightWalk {
    uint32_t max_depth, pass, path0, maxv;
    uint64_t seed;
    wr_path_vertex* out;
    uint32_t* counts;

    __device__ __forceinline__ bool begin(const SceneCtx& sc, uint32_t k, LaneStack& st, f3& o, f3& d,
                                          uint32_t& inside, uint32_t& contact) const {
        const uint32_t path = path0 + k;
        wr_path_vertex* V = out + (size_t)k * maxv;
        float rn[4];
        rng4(seed, path, pass, kLightVertex, rn);
        const LightSample L = sample_light(sc, rn);
        if (!L.ok) {  // the reference's empty-mesh light ray: no direction, radiance or contact, and it hits nothing
            const f3 z = mk(0.f, 0.f, 0.f);
            put_vertex(V[0], z, z, z, 1.f, 1.f, WR_NONE, 0u, WR_NONE, false);
            put_terminate(V[1], z);
            counts[k] = 2;
            return false;
        }
        rng4(seed, path, pass, kLightVertex + 1, rn);
        // UniformSphereSampler::sample (uniformSphereSampler.h:6-20)
        const float term1 = (float)(2.0 * kPi * (double)rn[0]);
        const float term2 = 2.f * sqrtf(rn[1] - rn[1] * rn[1]);
        d = mk(cosf(term1) * term2, 1.f - 2.f * rn[1], sinf(term1) * term2);
        float dp = (float)(kInvPi * 0.25f);
        if (dot(d, L.n) < 0.f) d = mk(-d.x, -d.y, -d.z);
        o = L.o;
        inside = find_inside(sc.S, o, d, L.obj, st);
        contact = L.obj;
        dp *= 2.f;
        put_vertex(V[0], o, d, L.rad, L.op, dp, L.obj, L.tri, inside, false);
        return true;
    }

    __device__ __forceinline__ bool step(const SceneCtx& sc, uint32_t k, uint32_t s, f3 o, f3 d, const PHit& hit,
                                         LaneStack& st, Out& r) const {
        wr_path_vertex* V = out + (size_t)k * maxv;
        counts[k] = s + 2;  // of a path that ends here; a later step overwrites it
        // an escaped ray ends the path at the origin before its own; the light
        // ray's hit counts only at dist > 0 (abstractObj.cpp:46)
        if (hit.rec == WR_NONE || (s == 0 && !(hit.t > 0.f))) {
            const float* e = V[s == 0 ? 0 : s - 1].origin;
            put_terminate(V[s + 1], mk(e[0], e[1], e[2]));
            return false;
        }
        const uint32_t inside = V[s].inside_obj;
        float rn[4];
        rng4(seed, path0 + k, pass, kLightVertex + 2 + s, rn);
        r = scatter(sc, inside != WR_NONE ? inside : hit.obj, o, d, hit, inside, rn, st);
        const bool absorbed = (double)len(r.d) < 0.5;
        if (!absorbed && s + 1 > max_depth) {
            put_terminate(V[s + 1], o);
            return false;
        }
        const uint32_t ctri = sc.S.tris[hit.rec].prim - sc.S.objs[hit.obj].prim_base;  // intersectTriangleID
        put_vertex(V[s + 1], r.o, r.d, r.rad, r.op, r.dp, r.contact, ctri, r.inside, r.delta);
        return !absorbed;
    }
};

// Light points of one path: vertices 1.. before the first emissive contact,
// without the delta ones.
__device__ __forceinline__ bool photon_at(const SceneDev& S, const wr_path_vertex& v, bool& stop) {
    stop = v.contact_obj != WR_NONE && S.objs[v.contact_obj].mat == WR_MAT_EMISSIVE;
    return !stop && !(v.flags & WR_VERTEX_DELTA);
}

__global__ __launch_bounds__(256) void k_photon_count(SceneDev S, const wr_path_vertex* V, const uint32_t* counts,
                                                      uint32_t n, uint32_t maxv, uint32_t* pc) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const uint32_t c = min(counts[k], maxv);
    uint32_t m = 0;
    for (uint32_t i = 1; i < c; i++) {
        bool stop;
        const bool keep = photon_at(S, V[(size_t)k * maxv + i], stop);
        if (stop) break;
        m += keep;
    }
    pc[k] = m;
}

__global__ __launch_bounds__(256) void k_photon_write(SceneDev S, const wr_path_vertex* V, const uint32_t* counts,
                                                      uint32_t n, uint32_t maxv, const uint64_t* offs,
                                                      uint64_t base, uint64_t cap, float* pos, uint32_t* src) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const uint32_t c = min(counts[k], maxv);
    uint64_t j = base + offs[k];
    for (uint32_t i = 1; i < c; i++) {
        const wr_path_vertex& v = V[(size_t)k * maxv + i];
        bool stop;
        const bool keep = photon_at(S, v, stop);
        if (stop) break;
        if (!keep) continue;
        if (j < cap) {
            pos[3 * j] = v.origin[0];
            pos[3 * j + 1] = v.origin[1];
            pos[3 * j + 2] = v.origin[2];
            src[2 * j] = k;
            src[2 * j + 1] = i;
        }
        j++;
    }
}

__global__ __launch_bounds__(256) void k_fill_leading(uint64_t n, uint64_t cap, float* pos, uint32_t* src) {
    for (uint64_t j = blockIdx.x * 256ull + threadIdx.x; j < n && j < cap; j += (uint64_t)gridDim.x * 256) {
        pos[3 * j] = 0.f;
        pos[3 * j + 1] = 0.f;
        pos[3 * j + 2] = 0.f;
        src[2 * j] = WR_NONE;
        src[2 * j + 1] = WR_NONE;
    }
}

// ---- hash grid ------------------------------------------------------------
// The grids of several passes are built together: every kernel below covers all
// blocks of points (segments), and one sort orders them by (segment, cell).
// Built one by one, the eight grids of a 256^2 PhotonMap call (1M points) took
// 1.6 ms in 190 launches, with two synchronisations each; now 0.18 ms in 12.
struct GridSegs {
    const uint32_t* starts;  // nullptr: one segment
    uint32_t lead, nseg, total;
    __device__ __forceinline__ uint32_t first(uint32_t b) const {
        return starts ? b * lead + starts[b] : (b ? total : 0u);
    }
    // the segment of point i
    __device__ __forceinline__ uint32_t of(uint32_t i) const {
        uint32_t lo = 0, hi = nseg;  // first(lo) <= i < first(hi)
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (first(mid) <= i) lo = mid;
            else hi = mid;
        }
        return lo;
    }
};

// Partial bounding boxes: `parts` workgroups per segment, their boxes in part
// (6 floats each).  No atomics: 13,000 of them on six words took most of the
// 155 us that 568,000 points' box took.
__global__ __launch_bounds__(256) void k_grid_bbox(GridSegs G, const float* pos, uint32_t parts, float* part) {
    const uint32_t b = blockIdx.x / parts, k = blockIdx.x % parts;
    const uint32_t end = G.first(b + 1);
    float mn[3] = {1e36f, 1e36f, 1e36f}, mx[3] = {-1e36f, -1e36f, -1e36f};
    for (uint64_t i = (uint64_t)G.first(b) + k * 256 + threadIdx.x; i < end; i += (uint64_t)parts * 256) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const float v = pos[3 * i + a];
            mn[a] = fminf(mn[a], v);
            mx[a] = fmaxf(mx[a], v);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        for (int off = 32; off > 0; off >>= 1) {
            mn[a] = fminf(mn[a], __shfl_xor(mn[a], off));
            mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off));
        }
    }
    __shared__ float wave[4][6];
    const uint32_t w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int a = 0; a < 3; a++) {
            wave[w][a] = mn[a];
            wave[w][3 + a] = mx[a];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = wave[0][threadIdx.x];
        for (int k2 = 1; k2 < 4; k2++)
            v = threadIdx.x < 3 ? fminf(v, wave[k2][threadIdx.x]) : fmaxf(v, wave[k2][threadIdx.x]);
        part[6 * (size_t)blockIdx.x + threadIdx.x] = v;
    }
}

// The view of every segment's grid, one wave per segment: its box from the
// partial ones, and the check that the integer cell coordinates stay
// representable.
__global__ __launch_bounds__(64) void k_grid_views(GridSegs G, const float* part, uint32_t parts,
                                                   const GridParams* params, uint32_t n_cells, const int* ends,
                                                   const uint32_t* idx, const float* sorted_pos, const uint32_t* src,
                                                   GridView* views, uint32_t* err) {
    const uint32_t b = blockIdx.x;
    float mn[3] = {1e36f, 1e36f, 1e36f}, mx[3] = {-1e36f, -1e36f, -1e36f};
    for (uint32_t k = threadIdx.x; k < parts; k += 64)
        for (int a = 0; a < 3; a++) {
            mn[a] = fminf(mn[a], part[6 * (size_t)(b * parts + k) + a]);
            mx[a] = fmaxf(mx[a], part[6 * (size_t)(b * parts + k) + 3 + a]);
        }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        for (int off = 32; off > 0; off >>= 1) {
            mn[a] = fminf(mn[a], __shfl_xor(mn[a], off));
            mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off));
        }
    }
    if (threadIdx.x != 0) return;
    const GridParams P = params[b];
    const size_t first = G.first(b);
    GridView v;
    bool fits = true;
    for (int a = 0; a < 3; a++) {
        v.g.bmin[a] = mn[a];
        v.g.bmax[a] = mx[a];
        fits = fits && (mx[a] - mn[a]) * P.inv < 2147483520.f;
    }
    v.g.inv = P.inv;
    v.g.r2 = P.r2;
    v.g.n_cells = n_cells;
    v.ends = ends + (size_t)b * n_cells;
    v.idx = idx + first;
    v.pos = sorted_pos + 3 * first;
    v.src = src ? src + 2 * first : nullptr;
    v.r = P.r;
    views[b] = v;
    if (!fits && G.first(b + 1) > first) *err = 1u;
}

// Each point's sort key (its segment, then its cell: GetCellIndex(Vec3f),
// hashgrid.hxx:180-190) and its index within the segment.
__global__ __launch_bounds__(256) void k_grid_keys(GridSegs G, const GridView* views, const float* pos, uint32_t* keys,
                                                   uint32_t* vals) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= G.total) return;
    const uint32_t b = G.of(i);
    const GridDev g = views[b].g;
    const float* p = pos + 3 * (size_t)i;
    const float dx = p[0] - g.bmin[0], dy = p[1] - g.bmin[1], dz = p[2] - g.bmin[2];
    keys[i] = b * g.n_cells + grid_hash(g, (int)floorf(g.inv * dx), (int)floorf(g.inv * dy), (int)floorf(g.inv * dz));
    vals[i] = i - G.first(b);
}

// From the sorted keys: the end of every cell (the entries of its segment with
// a key up to its own, by binary search: no counts, so no atomics and no scan
// of the cells) and the positions in the grid's order.
__global__ __launch_bounds__(256) void k_grid_finish(GridSegs G, const float* pos, const uint32_t* keys,
                                                     const uint32_t* idx, uint32_t n_cells, int* ends,
                                                     float* sorted_pos) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < G.nseg * n_cells) {
        uint32_t lo = 0, n = G.total;  // the first entry with a larger key
        while (n > 0) {
            const uint32_t half = n >> 1;
            if (keys[lo + half] <= i) {
                lo += half + 1;
                n -= half + 1;
            } else {
                n = half;
            }
        }
        ends[i] = (int)(lo - G.first(i / n_cells));
    }
    if (i < G.total) {
        const size_t from = (size_t)G.first(keys[i] / n_cells) + idx[i];
        for (int a = 0; a < 3; a++) sorted_pos[3 * (size_t)i + a] = pos[3 * from + a];
    }
}

// The bounding box of every kGridChunk entries, one workgroup each.
__global__ __launch_bounds__(256) void k_grid_boxes(uint32_t total, const float* sorted_pos, float* boxes) {
    static_assert(wr::kGridChunk == 256, "one lane per entry");
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    float v[6];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const bool in = i < total;
        const float x = in ? sorted_pos[3 * (size_t)i + a] : 0.f;
        v[a] = in ? x : 1e38f;
        v[3 + a] = in ? x : -1e38f;
        for (int off = 32; off > 0; off >>= 1) {
            v[a] = fminf(v[a], __shfl_xor(v[a], off));
            v[3 + a] = fmaxf(v[3 + a], __shfl_xor(v[3 + a], off));
        }
    }
    __shared__ float wave[4][6];
    if ((threadIdx.x & 63) == 0)
        for (int a = 0; a < 6; a++) wave[threadIdx.x >> 6][a] = v[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        float r = wave[0][threadIdx.x];
        for (int k = 1; k < 4; k++) r = threadIdx.x < 3 ? fminf(r, wave[k][threadIdx.x]) : fmaxf(r, wave[k][threadIdx.x]);
        boxes[6 * (size_t)blockIdx.x + threadIdx.x] = r;
    }
}

// Ranges longer than this are scanned by the whole wave, 64 points a step, one
// query at a time (a crowded cell, or one that shares a hash bucket with it).
constexpr int kLongRange = 64;

// Ranges longer than this hand their whole query to k_grid_query_wide (one
// workgroup per query), so that no wave walks such a range alone.
constexpr int kHugeRange = 2048;

// defer: [0] the number of deferred queries, then their indices.
__global__ __launch_bounds__(256) void k_grid_query(GridView G, const float* q, uint32_t nq, uint32_t cap, uint32_t* counts,
                                                    uint32_t* out, uint32_t* defer) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    const GridDev& g = G.g;
    const int* ends = G.ends;
    const uint32_t* idx = G.idx;
    const float* pos = G.pos;
    // every lane stays to the end: the long ranges are scanned by the whole wave
    bool valid = k < nq;
    f3 qp = mk(0.f, 0.f, 0.f);
    int p[6] = {0, 0, 0, 0, 0, 0};
    if (valid) {
        qp = mk(q[3 * k], q[3 * k + 1], q[3 * k + 2]);
        if (!query_corner(g, qp, p)) {
            counts[k] = 0;
            valid = false;
        } else {
            bool huge = false;
            for (int j = 0; j < 8; j++) {
                const uint32_t c = query_cell(g, p, j);
                huge = huge || ends[c] - (c == 0 ? 0 : ends[c - 1]) > kHugeRange;
            }
            if (huge) {  // k_grid_query_wide writes this query's list and count
                defer[1 + atomicAdd(defer, 1u)] = k;
                valid = false;
            }
        }
    }
    uint32_t m = 0;
    for (int j = 0; j < 8; j++) {  // the reference's cell order
        int a = 0, b = 0;
        if (valid) {
            const uint32_t c = query_cell(g, p, j);
            a = c == 0 ? 0 : ends[c - 1];
            b = ends[c];
        }
        const bool long_range = b - a > kLongRange;
        if (!long_range) {
            for (; a < b; a++) {
                if (grid_near(g, pos, qp, a)) {
                    if (m < cap) out[(size_t)k * cap + m] = idx[a];
                    m++;
                }
            }
        }
        // long ranges: the wave scans them one query at a time, in order, so the
        // points keep the serial loop's order in the output
        for (uint64_t pend = __ballot(long_range); pend != 0; pend &= pend - 1) {
            const uint32_t L = __ffsll((unsigned long long)pend) - 1;
            const f3 lq = mk(__shfl(qp.x, L), __shfl(qp.y, L), __shfl(qp.z, L));
            const int la = __shfl(a, L), lb = __shfl(b, L);
            const uint32_t lk = __shfl(k, L);
            uint32_t lm = __shfl(m, L);
            // sixteen 64-point steps per iteration: their loads are in flight together
            // (a single wave walks the whole range, so its loads in flight set the pace)
            for (int base = la; base < lb; base += 16 * 64) {
                bool hit[16];
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const int ai = base + 64 * u + (int)lane;
                    hit[u] = ai < lb && grid_near(g, pos, lq, ai);
                }
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const uint64_t hm = __ballot(hit[u]);
                    if (hit[u]) {
                        const uint32_t slot = lm + (uint32_t)__popcll(hm & below);
                        if (slot < cap) out[(size_t)lk * cap + slot] = idx[base + 64 * u + (int)lane];
                    }
                    lm += (uint32_t)__popcll(hm);
                }
            }
            if (lane == L) m = lm;
        }
    }
    if (valid) counts[k] = m;
}

// The deferred queries, one workgroup per query: the workgroup walks the
// query's 8 cells in the reference's order, in chunks of kGridChunk entries of
// the grid's order, and skips every chunk whose bounding box is out of reach (a
// long range is mostly points that have nothing in common but their bucket, or
// one coincident heap such as VCM's leading points).  The test is exact: the
// distance to the box is formed by the operations of the distance to a point,
// each of them monotone under rounding, from per-axis distances no larger than
// any of its points', so a chunk is skipped only if every point of it would
// fail.  256 chunks are tested at a time; the points of the ones left are
// tested one per lane, and a hit's slot is the query's count so far, the hits
// of the earlier waves (LDS) and its rank in its wave's ballot, which keeps the
// serial order.  Every loop bound is the same for the whole workgroup.  Point
// by point, 260,000 queries over 568,000 points of which 307,200 share a
// bucket took 566 us; now 15 us.
__global__ __launch_bounds__(256) void k_grid_query_wide(GridView G, const float* boxes, const float* q, uint32_t cap,
                                                         uint32_t* counts, uint32_t* out, const uint32_t* defer) {
    __shared__ uint64_t near[4];   // the chunks in reach, a bit each
    __shared__ uint32_t wcnt[4];
    const GridDev& g = G.g;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t nd = defer[0];
    for (uint32_t d = blockIdx.x; d < nd; d += gridDim.x) {
        const uint32_t k = defer[1 + d];
        const f3 qp = mk(q[3 * k], q[3 * k + 1], q[3 * k + 2]);
        int p[6];
        (void)query_corner(g, qp, p);  // inside the box: only such queries are deferred
        uint32_t m = 0;
        for (int j = 0; j < 8; j++) {
            const uint32_t c = query_cell(g, p, j);
            const int a = c == 0 ? 0 : G.ends[c - 1];
            const int b = G.ends[c];
            if (a >= b) continue;
            const uint32_t last = (uint32_t)(b - 1) / wr::kGridChunk;
            for (uint32_t c0 = (uint32_t)a / wr::kGridChunk; c0 <= last; c0 += 256) {
                const uint32_t ch = c0 + threadIdx.x;
                bool reach = false;
                if (ch <= last) {
                    const float* B = boxes + 6 * (size_t)ch;
                    const f3 dv = mk(fmaxf(fmaxf(B[0] - qp.x, qp.x - B[3]), 0.f),
                                     fmaxf(fmaxf(B[1] - qp.y, qp.y - B[4]), 0.f),
                                     fmaxf(fmaxf(B[2] - qp.z, qp.z - B[5]), 0.f));
                    const float dist = len(dv);
                    reach = dist * dist <= g.r2;
                }
                const uint64_t rm = __ballot(reach);
                if (lane == 0) near[wave] = rm;
                __syncthreads();
                for (uint32_t w = 0; w < 4; w++) {
                    for (uint64_t left = near[w]; left != 0; left &= left - 1) {
                        const uint32_t chunk = c0 + 64 * w + (uint32_t)__ffsll((unsigned long long)left) - 1;
                        const int ai = (int)(chunk * wr::kGridChunk + threadIdx.x);
                        const bool hit = ai >= a && ai < b && grid_near(g, G.pos, qp, ai);
                        const uint64_t hm = __ballot(hit);
                        if (lane == 0) wcnt[wave] = (uint32_t)__popcll(hm);
                        __syncthreads();
                        uint32_t before = 0, all = 0;
                        for (uint32_t v = 0; v < 4; v++) {
                            before += v < wave ? wcnt[v] : 0u;
                            all += wcnt[v];
                        }
                        if (hit) {
                            const uint32_t slot = m + before + (uint32_t)__popcll(hm & below);
                            if (slot < cap) out[(size_t)k * cap + slot] = G.idx[ai];
                        }
                        m += all;
                        __syncthreads();  // wcnt serves the next chunk
                    }
                }
                __syncthreads();  // near serves the next 256 chunks
            }
        }
        if (threadIdx.x == 0) counts[k] = m;
    }
}

// Clears one word with a kernel rather than a memset, so a caller may record
// the query sequence into a graph.
__global__ void k_clear_word(uint32_t* p) { *p = 0u; }

}  // namespace wrd

// Deferred-query work list of wr_hashgrid_query_noalloc: the counter, then up
// to WR_HASHGRID_NOALLOC_MAX_QUERIES query indices (16 MiB per GPU, held until
// the process ends).  Host code never passes this name to a kernel: it uses
// the per-device address from hipGetSymbolAddress (noalloc_ptr below).
static __device__ __align__(256) uint32_t scratch[WR_HASHGRID_NOALLOC_MAX_QUERIES + 1];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
uint32_t* g_scratch_ptr[kMaxScratchDevices] = {};  // device address of scratch, per device
}  // namespace

namespace wr {
// Looks up scratch's address on `device`, which must be current.  Called once
// per device, from wr_ctx_create.
hipError_t noalloc_scratch_init(int device) {
    if (device < 0 || device >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return hipSuccess;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = (uint32_t*)p;
    return hipSuccess;
}

static uint32_t* noalloc_ptr(int device) {
    if (device < 0 || device >= kMaxScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_ptr[device];
}
}  // namespace wr


using namespace wrd;
using wr::fail;
using wr::hip_fail;

#define PH_CHECK(call, what)                         \
    do {                                             \
        hipError_t e_ = (call);                      \
        if (e_ != hipSuccess) return hip_fail(ctx, e_, what); \
    } while (0)

namespace wr {

hipError_t build_grids(wr_ctx* ctx, Scratch& mem, const float* d_pos, const uint32_t* d_src, uint64_t total,
                       const uint32_t* starts, uint32_t lead, uint32_t nseg, uint32_t n_cells,
                       const GridParams* params, GridView* views, uint32_t* err, float** boxes, float* sorted) {
    hipStream_t st = ctx->stream;
    const uint32_t cells = nseg * n_cells;
    // workgroups of 256 per segment's box: one per 1,024 points, at most 128
    const uint32_t parts = (uint32_t)std::min<uint64_t>(128, std::max<uint64_t>(1, total / nseg / 1024));
    int end_bit = 1;
    while (end_bit < 32 && (cells - 1) >> end_bit) end_bit++;
    size_t tb = 0;
    hipError_t e = hipSuccess;
    if (total)
        e = hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                               (uint32_t*)nullptr, (int)total, 0, end_bit, st);
    if (e != hipSuccess) return e;
    // what the grids keep, and what the build alone needs
    int* ends;
    uint32_t* idx;
    float* pos = sorted;
    if ((e = mem.get(&ends, sizeof(int) * (size_t)cells)) != hipSuccess) return e;
    if ((e = mem.get(&idx, sizeof(uint32_t) * total)) != hipSuccess) return e;
    if (!pos && (e = mem.get(&pos, sizeof(float) * 3 * total)) != hipSuccess) return e;
    if (boxes && (e = mem.get(boxes, sizeof(float) * 6 * ((total + kGridChunk - 1) / kGridChunk))) != hipSuccess)
        return e;
    Scratch sc(*ctx->pool);
    float* part;
    GridParams* d_params;
    uint32_t* keys;
    void* tmp;
    const size_t n4 = sizeof(uint32_t) * total;
    if ((e = sc.get(&part, sizeof(float) * 6 * (size_t)nseg * parts)) != hipSuccess) return e;
    if ((e = sc.get(&d_params, sizeof(GridParams) * nseg)) != hipSuccess) return e;
    if ((e = sc.get(&keys, 3 * n4)) != hipSuccess) return e;
    if ((e = sc.get(&tmp, tb)) != hipSuccess) return e;
    uint32_t *sorted_keys = keys + total, *vals = sorted_keys + total;
    if ((e = hipMemcpyAsync(d_params, params, sizeof(GridParams) * nseg, hipMemcpyHostToDevice, st)) != hipSuccess)
        return e;
    const GridSegs G{starts, lead, nseg, (uint32_t)total};
    k_grid_bbox<<<nseg * parts, 256, 0, st>>>(G, d_pos, parts, part);
    k_grid_views<<<nseg, 64, 0, st>>>(G, part, parts, d_params, n_cells, ends, idx, pos, d_src, views, err);
    const uint32_t blocks = (uint32_t)((total + 255) / 256);
    if (total) {
        k_grid_keys<<<blocks, 256, 0, st>>>(G, views, d_pos, keys, vals);
        // stable: points of one cell keep their input order, as the serial scatter does
        e = hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, sorted_keys, vals, idx, (int)total, 0, end_bit, st);
        if (e != hipSuccess) return e;
    }
    const uint32_t most = (uint32_t)std::max<uint64_t>(total, cells);
    k_grid_finish<<<(most + 255) / 256, 256, 0, st>>>(G, d_pos, sorted_keys, idx, n_cells, ends, pos);
    if (boxes && total) k_grid_boxes<<<blocks, 256, 0, st>>>((uint32_t)total, pos, *boxes);
    return hipGetLastError();
}

}  // namespace wr

extern "C" {

int wr_light_paths(wr_ctx* ctx, const wr_scene* s, uint32_t max_depth, uint64_t seed, uint32_t pass, uint32_t path0,
                   uint32_t n_paths, uint32_t max_vertices, wr_path_vertex* d_vertices, uint32_t* d_counts) {
    if (!ctx || !s || (n_paths && (!d_vertices || !d_counts))) return fail(ctx, WR_EINVAL, "wr_light_paths: bad argument");
    if (!s->built) return fail(ctx, WR_ESTATE, "wr_light_paths: scene not built");
    if ((uint64_t)max_vertices < (uint64_t)max_depth + 3)
        return fail(ctx, WR_EINVAL, "wr_light_paths: max_vertices must be at least max_depth + 3");
    if ((uint64_t)path0 + n_paths > 0x100000000ull) return fail(ctx, WR_EINVAL, "wr_light_paths: path ids overflow");
    if (n_paths == 0) return WR_OK;
    (void)hipSetDevice(ctx->device);
    const LightWalk P{max_depth, pass, path0, max_vertices, seed, d_vertices, d_counts};
    PH_CHECK(wr::run_walk(ctx, s->dev, s->hdrs[0], P, n_paths, max_depth + 1), "wr_light_paths");
    PH_CHECK(hipStreamSynchronize(ctx->stream), "wr_light_paths");
    return WR_OK;
}

int wr_photons_collect(wr_ctx* ctx, const wr_scene* s, const wr_path_vertex* d_vertices, const uint32_t* d_counts,
                       uint32_t n_paths, uint32_t max_vertices, uint64_t n_leading, float* d_pos, uint32_t* d_src,
                       uint64_t cap, uint64_t* n_out) {
    if (!ctx || !s || !n_out || (cap && (!d_pos || !d_src)) || (n_paths && (!d_vertices || !d_counts)))
        return fail(ctx, WR_EINVAL, "wr_photons_collect: bad argument");
    if (!s->built) return fail(ctx, WR_ESTATE, "wr_photons_collect: scene not built");
    if (n_paths >= (1u << 31)) return fail(ctx, WR_EINVAL, "wr_photons_collect: too many paths");
    (void)hipSetDevice(ctx->device);
    hipStream_t st = ctx->stream;
    wr::Scratch sc(*ctx->pool);
    uint32_t* pc = nullptr;
    uint64_t* offs = nullptr;
    PH_CHECK(sc.get(&pc, sizeof(uint32_t) * (n_paths + 1)), "hipMalloc(photons)");
    PH_CHECK(sc.get(&offs, sizeof(uint64_t) * (n_paths + 1)), "hipMalloc(photons)");
    uint64_t total = 0;
    if (n_paths) {
        const uint32_t blocks = (n_paths + 255) / 256;
        k_photon_count<<<blocks, 256, 0, st>>>(s->dev, d_vertices, d_counts, n_paths, max_vertices, pc);
        PH_CHECK(hipGetLastError(), "wr_photons_collect");
        // exclusive offsets over n_paths + 1 entries (the last one is the total)
        PH_CHECK(hipMemsetAsync(pc + n_paths, 0, sizeof(uint32_t), st), "wr_photons_collect");
        size_t tb = 0;
        PH_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, pc, offs, (int)n_paths + 1, st), "hipcub scan");
        void* tmp = nullptr;
        PH_CHECK(sc.get(&tmp, tb), "hipMalloc(photons)");
        PH_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, tb, pc, offs, (int)n_paths + 1, st), "hipcub scan");
        PH_CHECK(hipMemcpyAsync(&total, offs + n_paths, sizeof(uint64_t), hipMemcpyDeviceToHost, st),
                 "wr_photons_collect");
        k_photon_write<<<blocks, 256, 0, st>>>(s->dev, d_vertices, d_counts, n_paths, max_vertices, offs, n_leading,
                                                cap, d_pos, d_src);
        PH_CHECK(hipGetLastError(), "wr_photons_collect");
    }
    if (n_leading && cap) {
        const uint64_t m = std::min(n_leading, cap);
        k_fill_leading<<<(unsigned)std::min<uint64_t>((m + 255) / 256, 65535), 256, 0, st>>>(n_leading, cap, d_pos,
                                                                                             d_src);
        PH_CHECK(hipGetLastError(), "wr_photons_collect");
    }
    PH_CHECK(hipStreamSynchronize(st), "wr_photons_collect");
    *n_out = n_leading + total;
    return WR_OK;
}

int wr_hashgrid_build(wr_ctx* ctx, const float* d_pos, uint64_t n, float radius, uint32_t n_cells,
                      wr_hashgrid** out) {
    if (!ctx || !out || (n && !d_pos) || n_cells == 0) return fail(ctx, WR_EINVAL, "wr_hashgrid_build: bad argument");
    *out = nullptr;
    if (n >= (1ull << 31)) return fail(ctx, WR_EINVAL, "wr_hashgrid_build: too many points");
    if (!(radius > 0.f) || !std::isfinite(radius)) return fail(ctx, WR_EINVAL, "wr_hashgrid_build: radius must be > 0");
    (void)hipSetDevice(ctx->device);
    hipStream_t st = ctx->stream;
    std::unique_ptr<wr_hashgrid> g(new wr_hashgrid);
    g->ctx = ctx;
    g->pool = ctx->pool;
    g->mem.reset(new wr::Scratch(*g->pool));
    g->n = n;
    // Build with aMaxDist = 0: mCellSize = 2 * radius (hashgrid.hxx:28-35)
    float max_dist = 0.f;
    if (std::fabs(max_dist) < 1e-5) max_dist = radius;
    const float cell = max_dist * 2.f;
    const GridParams P{1.f / cell, radius * radius, radius};
    wr::Scratch sc(*ctx->pool);
    GridView* view = nullptr;
    float* boxes = nullptr;
    struct {
        GridView v;
        uint32_t err;
    } back;
    PH_CHECK(sc.get(&view, sizeof(back)), "hipMalloc(hashgrid)");
    uint32_t* err = (uint32_t*)((char*)view + ((char*)&back.err - (char*)&back));
    k_clear_word<<<1, 1, 0, st>>>(err);
    PH_CHECK(wr::build_grids(ctx, *g->mem, d_pos, nullptr, n, nullptr, 0, 1, n_cells, &P, view, err, &boxes),
             "wr_hashgrid_build");
    PH_CHECK(hipMemcpyAsync(&back, view, sizeof(back), hipMemcpyDeviceToHost, st), "wr_hashgrid_build");
    PH_CHECK(hipStreamSynchronize(st), "wr_hashgrid_build");
    if (back.err)
        return fail(ctx, WR_EINVAL, "wr_hashgrid_build: too many cells across the points' box for this radius");
    g->v = back.v;
    g->boxes = boxes;
    *out = g.release();
    return WR_OK;
}

int wr_hashgrid_export(const wr_hashgrid* g, float* bbox, int32_t* cell_ends, int32_t* indices) {
    if (!g) return fail(nullptr, WR_EINVAL, "wr_hashgrid_export: grid is NULL");
    wr_ctx* ctx = g->ctx;
    (void)hipSetDevice(ctx->device);
    if (bbox)
        for (int a = 0; a < 3; a++) {
            bbox[a] = g->v.g.bmin[a];
            bbox[3 + a] = g->v.g.bmax[a];
        }
    if (cell_ends)
        PH_CHECK(hipMemcpy(cell_ends, g->v.ends, sizeof(int) * g->v.g.n_cells, hipMemcpyDeviceToHost), "wr_hashgrid_export");
    if (indices && g->n)
        PH_CHECK(hipMemcpy(indices, g->v.idx, sizeof(uint32_t) * g->n, hipMemcpyDeviceToHost), "wr_hashgrid_export");
    return WR_OK;
}

int wr_hashgrid_query(wr_hashgrid* g, const float* d_queries, uint64_t nq, uint32_t cap, uint32_t* d_counts,
                      uint32_t* d_idx) {
    if (!g || (nq && (!d_queries || !d_counts)) || (cap && nq && !d_idx))
        return fail(g ? g->ctx : nullptr, WR_EINVAL, "wr_hashgrid_query: bad argument");
    wr_ctx* ctx = g->ctx;
    if (nq >= (1ull << 32)) return fail(ctx, WR_EINVAL, "wr_hashgrid_query: too many queries");
    if (nq == 0) return WR_OK;
    (void)hipSetDevice(ctx->device);
    if (g->defer_cap < nq + 1) {
        g->pool->put(g->defer);
        g->defer = nullptr;
        g->defer_cap = 0;
        PH_CHECK(g->pool->get(&g->defer, sizeof(uint32_t) * (nq + 1)), "hipMalloc(hashgrid query)");
        g->defer_cap = nq + 1;
    }
    PH_CHECK(hipMemsetAsync(g->defer, 0, sizeof(uint32_t), ctx->stream), "wr_hashgrid_query");
    k_grid_query<<<(unsigned)((nq + 255) / 256), 256, 0, ctx->stream>>>(g->v, d_queries, (uint32_t)nq, cap, d_counts,
                                                                         d_idx, g->defer);
    PH_CHECK(hipGetLastError(), "wr_hashgrid_query");
    // the deferred queries: a workgroup each, as many workgroups as fill the device twice
    const unsigned wide_grid = (unsigned)std::min<uint64_t>(nq, 2048);
    k_grid_query_wide<<<wide_grid, 256, 0, ctx->stream>>>(g->v, g->boxes, d_queries, cap, d_counts, d_idx, g->defer);
    PH_CHECK(hipGetLastError(), "wr_hashgrid_query");
    PH_CHECK(hipStreamSynchronize(ctx->stream), "wr_hashgrid_query");
    return WR_OK;
}

int wr_hashgrid_query_noalloc(wr_hashgrid* g, const float* d_queries, uint64_t nq, uint32_t cap, uint32_t* d_counts,
                              uint32_t* d_idx) {
    if (!g || (nq && (!d_queries || !d_counts)) || (cap && nq && !d_idx))
        return fail(g ? g->ctx : nullptr, WR_EINVAL, "wr_hashgrid_query_noalloc: bad argument");
    wr_ctx* ctx = g->ctx;
    if (nq > WR_HASHGRID_NOALLOC_MAX_QUERIES)
        return fail(ctx, WR_EINVAL, "wr_hashgrid_query_noalloc: more than WR_HASHGRID_NOALLOC_MAX_QUERIES (4,194,304) "
                                    "queries; use wr_hashgrid_query or split the call");
    if (nq == 0) return WR_OK;
    PH_CHECK(hipSetDevice(ctx->device), "wr_hashgrid_query_noalloc");
    uint32_t* defer = wr::noalloc_ptr(ctx->device);
    if (!defer) return fail(ctx, WR_ESTATE, "wr_hashgrid_query_noalloc: work list not set up on this device");
    // the list keeps the previous call's contents: only its counter must start at zero
    k_clear_word<<<1, 1, 0, ctx->stream>>>(defer);
    PH_CHECK(hipGetLastError(), "wr_hashgrid_query_noalloc");
    k_grid_query<<<(unsigned)((nq + 255) / 256), 256, 0, ctx->stream>>>(g->v, d_queries, (uint32_t)nq, cap, d_counts,
                                                                         d_idx, defer);
    PH_CHECK(hipGetLastError(), "wr_hashgrid_query_noalloc");
    const unsigned wide_grid = (unsigned)std::min<uint64_t>(nq, 2048);
    k_grid_query_wide<<<wide_grid, 256, 0, ctx->stream>>>(g->v, g->boxes, d_queries, cap, d_counts, d_idx, defer);
    PH_CHECK(hipGetLastError(), "wr_hashgrid_query_noalloc");
    return WR_OK;
}

void wr_hashgrid_destroy(wr_hashgrid* g) {
    if (!g) return;
    (void)hipSetDevice(g->pool->device);
    g->pool->put(g->defer);
    g->mem.reset();
    delete g;
}

}  // extern "C"
