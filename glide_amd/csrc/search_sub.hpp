// What the host side of the per-partition search and its kernels share; compiled once per degree bucket like search.hpp's.
#pragma once
#include "beam.hpp"

namespace glide {

struct SubArgs {
    const float* data;          // the staged partition
    const uint32_t* graph;      // partition-local ids
    const uint32_t* map;        // local id -> original id
    const float* queries;
    const uint32_t* segment_ids;
    const uint32_t* query_list;   // nullable: the queries that selected this partition (then segment_ids is not read)
    // pair mode (nullable pair_segment): block p searches query query_list[p] in partition pair_segment[p]; data / graph /
    // map are then the arrays of all partitions, addressed through segment_starts, and the beam head goes to pair_dists / pair_ids
    const uint32_t* pair_segment;
    const uint32_t* segment_starts;
    const uint32_t* segment_start_points;
    float* pair_dists;
    uint32_t* pair_ids;
    uint32_t* final_ids;
    float* final_dists;
    unsigned long long* counters;
    uint32_t query_num, centroid_num, segment_id, start_point, top_k, max_topk, list_len;
    BeamParams p;
};

using sub_fn = void (*)(SubArgs);

sub_fn pick_sub_64(uint32_t beam, uint32_t dim);
sub_fn pick_sub_128(uint32_t beam, uint32_t dim);
sub_fn pick_sub_256(uint32_t beam, uint32_t dim);
inline sub_fn pick_sub(uint32_t degree, uint32_t beam, uint32_t dim) {
    return degree <= 64 ? pick_sub_64(beam, dim) : degree <= 128 ? pick_sub_128(beam, dim) : pick_sub_256(beam, dim);
}

}  // namespace glide
