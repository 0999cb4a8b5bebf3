// What the host side of glide_hip_search and its kernels share.  The kernels are compiled once per degree bucket
// (search_kernels.hip with GLIDE_CAND = 64, 128, 256), so that the buckets compile side by side.
#pragma once
#include "beam.hpp"

namespace glide {

struct SearchArgs {
    const float* data;
    const uint32_t* graph;
    const float* centroids;
    const uint32_t* start_points;
    const float* queries;
    uint32_t* result_ids;
    float* result_dists;
    unsigned long long* counters;
    uint32_t centroid_num, max_centroid, top_k, query_num;
    BeamParams p;
    const unsigned char* bytes;   // the rows as bytes, for the kernels for rows of bytes
};

// Wavefronts of a team (search_team_kernel) and what one needs.
constexpr int kTeam = 4;

template <int DIMV>
struct TeamShape {
    static constexpr int U = DIMV >= 16 ? 1 : (DIMV == 8 ? 2 : 4);   // row steps in flight per wavefront: 64 row registers either way
    static constexpr size_t query_bytes = sizeof(float4) * RowShape<DIMV>::NV * RowShape<DIMV>::LPR;
};

using search_fn = void (*)(SearchArgs);

// The kernel for a beam and a row length; one function per degree bucket.
search_fn pick_search_64(uint32_t beam, uint32_t dim, bool team);
search_fn pick_search_128(uint32_t beam, uint32_t dim, bool team);
search_fn pick_search_256(uint32_t beam, uint32_t dim, bool team);
// Rows of bytes, up to 64 slots and kMostByteDims dims: the queries of bytes, and the fp32 kernel for those left over.
search_fn pick_search_bytes(uint32_t beam, uint32_t dim);
search_fn pick_search_left_over(uint32_t beam, uint32_t dim);

}  // namespace glide
