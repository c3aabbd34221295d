// merge_entry.h -- one entry of VCMTracer's merge queue (bdpt.hip).
//
// Word 0 names an eye vertex, word 1 a light point.  The eye vertex i of lane
// (pixel and pass) `lane` is record lane * maxv + i of the eye sub-paths, maxv
// records each: wr_render_vcm keeps lanes * maxv below 2^31, so the index fits
// one word at every image size and path length that it takes (a lane and a
// vertex in fixed bits of a word do not: images have 2^24 lanes and more).
#pragma once
#include <cstdint>

namespace wr {

constexpr uint32_t merge_entry(uint32_t lane, uint32_t vertex, uint32_t maxv) { return lane * maxv + vertex; }
constexpr uint32_t merge_lane(uint32_t entry, uint32_t maxv) { return entry / maxv; }
constexpr uint32_t merge_vertex(uint32_t entry, uint32_t maxv) { return entry % maxv; }

}  // namespace wr
