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
    const unsigned char* bytes;   // pair mode: the rows as bytes, for the kernels for rows of bytes,
    const uint32_t* other;        // and whether some row is not of bytes after all
};

using sub_fn = void (*)(SubArgs);

sub_fn pick_sub_64(uint32_t beam, uint32_t dim, bool six);
sub_fn pick_sub_128(uint32_t beam, uint32_t dim, bool six);
sub_fn pick_sub_256(uint32_t beam, uint32_t dim, bool six);

// Rows of bytes, pair mode, up to 64 slots and kMostByteDims dims: the pairs whose query is of bytes, and the fp32 kernel for
// those left over.
sub_fn pick_sub_bytes(uint32_t beam, uint32_t dim);
sub_fn pick_sub_left_over(uint32_t beam, uint32_t dim);

size_t simd_count();   // of the current device; 0 if it cannot be told

// Whether a launch of this many wavefronts runs with six rather than five per SIMD where the kernel comes in both forms
// (beams up to 64).  The searches of a full chip take longer about in proportion to their number, so what counts is how well
// the launch fills its last round: six where rounds times residency is a tenth less.  Measured at beam 64, five against six:
// 5 193 pairs over 1.2M x 96 unit rows 737 / 586 us, 5 453 over 1M x 128 byte rows 939 / 790 us, 10 366 over the unit rows
// 1 155 / 1 037 us; the other way round 12 440 over 60k byte rows 1 021 / 1 120 us and 13 770 over the million 1 747 / 1 779 us.
// With many rounds the last one counts for little, and partitions that do not stay in cache, bound by their gathers, run
// better with five (52 919 over 250k byte rows 3 963 / 4 214 us).
inline bool six_resident(uint32_t wavefronts) {
    const size_t simds = simd_count();
    if (simds == 0) return false;
    const size_t five = (wavefronts + 5 * simds - 1) / (5 * simds) * 5, six = (wavefronts + 6 * simds - 1) / (6 * simds) * 6;
    return six * 10 <= five * 9;
}
inline sub_fn pick_sub(uint32_t degree, uint32_t beam, uint32_t dim, uint32_t wavefronts) {
    const bool six = degree <= 64 && beam <= 64 && dim <= 512 && six_resident(wavefronts);
    return degree <= 64 ? pick_sub_64(beam, dim, six) : degree <= 128 ? pick_sub_128(beam, dim, six) : pick_sub_256(beam, dim, six);
}

}  // namespace glide
