// What the host side of the graph construction and its per-point kernels share; the kernels are compiled once per degree
// bucket (graph_kernels.hip with GLIDE_CAND = 64, 128, 256).
#pragma once
#include "prune.hpp"

namespace glide {

struct BuildArgs {
    const float* reorder_data;
    const uint32_t* knn_graph;
    const uint32_t* map;
    const uint32_t* segment_starts;
    const uint32_t* segment_lengths;
    const uint32_t* start_points;
    uint32_t* graph;
    unsigned long long* counters;
    uint32_t first_point, point_count;   // reorder ids [first_point, first_point + point_count)
    uint32_t segment_num, graph_degree;
    uint32_t boundary_start;             // boundary kernel: segment start (= num); 0xffffffff for the regular kernel
    uint32_t boundary_start_point;
    float relaxant;
    BeamParams p;                         // p.degree = knn_degree
    const unsigned char* bytes;           // the same rows as bytes; the kernels for rows of bytes read nothing else
    const unsigned char* rough;           // the same rows in fp16 (glide_hip_pack_rough_rows), for the kernels that look at them first
};

struct RefineArgs {
    const float* data;
    const uint32_t* graph_in;
    uint32_t* graph_out;
    const float* centroids;
    const uint32_t* start_points;
    unsigned long long* counters;
    const uint32_t* order;   // nullable: workgroup i refines point order[i] (a permutation of the points)
    uint32_t num, centroid_num, max_centroid, segment_start_point;
    float relaxant;
    BeamParams p;   // p.degree = graph_degree
    const unsigned char* bytes;   // the same rows as bytes, for the kernels for rows of bytes
    const unsigned char* rough;   // the same rows in fp16, for the kernels that look at them first
};

using build_fn = void (*)(BuildArgs);
using refine_fn = void (*)(RefineArgs);

build_fn pick_build_64(uint32_t beam, uint32_t dim);
build_fn pick_build_128(uint32_t beam, uint32_t dim);
build_fn pick_build_256(uint32_t beam, uint32_t dim);
refine_fn pick_refine_64(uint32_t beam, uint32_t dim);
refine_fn pick_refine_128(uint32_t beam, uint32_t dim);
refine_fn pick_refine_256(uint32_t beam, uint32_t dim);
// rows of bytes: up to 64 slots (kNN degree; graph degree) and kMostByteDims dims
build_fn pick_build_bytes(uint32_t beam, uint32_t dim);
refine_fn pick_refine_bytes(uint32_t beam, uint32_t dim);
// rows looked at in fp16 first: up to 64 slots, beams up to kMostRoughBeam
constexpr uint32_t kMostRoughDims = 1024, kMostRoughBeam = 128;
build_fn pick_build_rough(uint32_t beam, uint32_t dim);
refine_fn pick_refine_rough(uint32_t beam, uint32_t dim);
inline build_fn pick_build(uint32_t degree, uint32_t beam, uint32_t dim) {
    return degree <= 64 ? pick_build_64(beam, dim) : degree <= 128 ? pick_build_128(beam, dim) : pick_build_256(beam, dim);
}
inline refine_fn pick_refine(uint32_t degree, uint32_t beam, uint32_t dim) {
    return degree <= 64 ? pick_refine_64(beam, dim) : degree <= 128 ? pick_refine_128(beam, dim) : pick_refine_256(beam, dim);
}

}  // namespace glide
