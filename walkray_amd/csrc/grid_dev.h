// grid_dev.h -- the photon hash grid (HashGrid, hashgrid.hxx:15-203) as the
// device sees it: its parameters, the cell hash, the query's eight cells and
// the distance test, shared by the grid kernels (photon.hip) and the vertex
// merging of VCMTracer (bdpt.hip); and the library's grid handle.
#pragma once
#include <hip/hip_runtime.h>

#include "pt_dev.h"
#include "wr_capi_internal.h"

#pragma clang fp contract(off)

namespace wrd {

struct GridDev {
    float bmin[3], bmax[3];
    float inv;     // mInvCellSize
    float r2;      // mRadius * mRadius
    uint32_t n_cells;
};

// GetCellIndex(Vec3i) (hashgrid.hxx:170-178)
__device__ __forceinline__ uint32_t grid_hash(const GridDev& g, int cx, int cy, int cz) {
    const uint32_t x = (uint32_t)cx, y = (uint32_t)cy, z = (uint32_t)cz;
    return ((x * 73856093u) ^ (y * 19349663u) ^ (z * 83492791u)) % g.n_cells;
}

// The distance test of HashGrid::Process (hashgrid.hxx:142-147): |q - p|^2 <= r^2,
// p the a-th point in the grid's order.
__device__ __forceinline__ bool grid_near(const GridDev& g, const float* sorted_pos, f3 qp, int a) {
    const float* p = sorted_pos + 3 * (size_t)a;
    const f3 dv = mk(qp.x - p[0], qp.y - p[1], qp.z - p[2]);
    const float dist = len(dv);
    return dist * dist <= g.r2;
}

// The query's cell corner and its nearer neighbours (HashGrid::Process); false
// outside the grid's box.
__device__ __forceinline__ bool query_corner(const GridDev& g, f3 qp, int p[6]) {
    const f3 dmin = mk(qp.x - g.bmin[0], qp.y - g.bmin[1], qp.z - g.bmin[2]);
    const f3 dmax = mk(g.bmax[0] - qp.x, g.bmax[1] - qp.y, g.bmax[2] - qp.z);
    if (dmin.x < 0.f || dmin.y < 0.f || dmin.z < 0.f || dmax.x < 0.f || dmax.y < 0.f || dmax.z < 0.f) return false;
    const f3 cp = mk(g.inv * dmin.x, g.inv * dmin.y, g.inv * dmin.z);
    const f3 cf = mk(floorf(cp.x), floorf(cp.y), floorf(cp.z));
    p[0] = (int)cf.x;
    p[1] = (int)cf.y;
    p[2] = (int)cf.z;
    p[3] = p[0] + (cp.x - cf.x < 0.5f ? -1 : +1);
    p[4] = p[1] + (cp.y - cf.y < 0.5f ? -1 : +1);
    p[5] = p[2] + (cp.z - cf.z < 0.5f ? -1 : +1);
    return true;
}

// Cell j of the query's 8, in the reference's order.
__device__ __forceinline__ uint32_t query_cell(const GridDev& g, const int p[6], int j) {
    return grid_hash(g, (j & 4) ? p[3] : p[0], (j & 2) ? p[4] : p[1], (j & 1) ? p[5] : p[2]);
}

// One grid as its users see it.  pos holds the positions in the grid's order
// (mIndices), so that a cell's points are read next to each other and their
// indices only where a point is in reach.
struct GridView {
    GridDev g;
    const int* ends;      // mCellEnds (n_cells)
    const uint32_t* idx;  // mIndices
    const float* pos;     // 3 floats per entry of idx
    const uint32_t* src;  // the caller's: 2 words per point (nullptr: none)
    float r;
};

// What the host knows of a grid before its points.
struct GridParams {
    float inv, r2, r;
};

}  // namespace wrd

namespace wr {
// Builds `nseg` grids of n_cells cells each over consecutive blocks of points
// in one go (photon.hip).  Block b starts at point b * lead + starts[b]
// (starts: nseg + 1 device words; nullptr with one block of all the points) and
// its grid has the parameters params[b] (host).  `total` points in all (below
// 2^31), nseg * n_cells below 2^31.  Enqueued on the context's stream: views
// (nseg device records) describe the grids in buffers taken from mem; *err (a
// zeroed device word) is set if a grid has too many cells across.  boxes
// (nullable): the bounding box of every kGridChunk entries of the order.
// sorted (nullable): where the positions in the grids' order go (3 * total
// floats; nullptr: into a buffer from mem).
constexpr uint32_t kGridChunk = 256;
hipError_t build_grids(wr_ctx* ctx, Scratch& mem, const float* d_pos, const uint32_t* d_src, uint64_t total,
                       const uint32_t* starts, uint32_t lead, uint32_t nseg, uint32_t n_cells,
                       const wrd::GridParams* params, wrd::GridView* views, uint32_t* err, float** boxes,
                       float* sorted = nullptr);
}  // namespace wr

// A built grid: mCellEnds (inclusive ends per cell), mIndices and the positions
// in its order, in buffers of the context's pool.
struct wr_hashgrid {
    wr_ctx* ctx = nullptr;
    std::shared_ptr<wr::WorkPool> pool;
    std::unique_ptr<wr::Scratch> mem;
    wrd::GridView v{};
    const float* boxes = nullptr;  // per kGridChunk entries of the order: min xyz, max xyz
    uint64_t n = 0;
    uint32_t* defer = nullptr;     // query calls: deferred-query counter and list (grown on demand)
    uint64_t defer_cap = 0;        // entries of defer
};
