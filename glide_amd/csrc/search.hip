// glide_hip_search: one query per wavefront beam search over the finished index.
// Reference: search_kernel (search_kernel.cuh:393-490) launched by GLIDE::search (glide_impl.cuh:370-454).
#include "search.hpp"
#include "host_util.hpp"

namespace glide {

size_t simd_count() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 0;
    return static_cast<size_t>(cus) * 4;
}

// One workgroup per query, up to half of what a launch can hold (2^32 threads); beyond that a wavefront takes several.
// Batches above what the chip holds at once are left to the hardware's dispatch.  Dividing them into equal rounds, several
// queries a wavefront, helps while rows come from memory and the rounds just fit what is resident (7 000 queries at beam
// 64: 743 against 633 us on unit rows), but rows that stay in cache make queries unequally long and lose by it (same batch
// on the mixture: 439 against 512 us; 25 000 queries in rounds of 6 250: 1.40 times the time there, 1.20 on rows from memory).
constexpr uint32_t kMostWorkgroups = 1u << 25;

}  // namespace glide

using namespace glide;

namespace {
int launch_search(const float* data, const unsigned char* bytes, uint32_t num, uint32_t dim, const uint32_t* graph, uint32_t graph_degree, const float* centroids,
                  uint32_t centroid_num, bool rank_all_centroids, const uint32_t* start_points, const float* queries, uint32_t query_num,
                  uint32_t top_k, uint32_t beam, uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                  uint32_t hash_reset_interval, int metric, uint32_t* result_ids, float* result_dists, unsigned long long* counters,
                  void* stream) {
    if (!data || !graph || !centroids || !start_points || !queries || !result_ids || !result_dists) return GLIDE_ERR_BAD_ARGUMENT;
    if (num == 0 || dim == 0 || graph_degree == 0 || centroid_num == 0 || beam == 0 || top_k == 0 || max_iterations == 0)
        return GLIDE_ERR_BAD_ARGUMENT;
    if (metric != GLIDE_METRIC_EUCLIDEAN && metric != GLIDE_METRIC_COSINE) return GLIDE_ERR_BAD_ARGUMENT;
    if (query_num == 0) return GLIDE_OK;
    if (graph_degree > 256 || !beam_supported(beam) || centroid_num > 256 || dim % 4 != 0 || dim > 4096 || top_k > beam ||
        hash_bit < 1 || hash_bit > 13)
        return GLIDE_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(data) % 16 || reinterpret_cast<uintptr_t>(queries) % 16 ||
        reinterpret_cast<uintptr_t>(centroids) % 16)
        return GLIDE_ERR_BAD_ARGUMENT;

    SearchArgs a;
    a.data = data;
    a.bytes = nullptr;
    a.graph = graph;
    a.centroids = centroids;
    a.start_points = start_points;
    a.queries = queries;
    a.result_ids = result_ids;
    a.result_dists = result_dists;
    a.counters = counters;
    a.centroid_num = centroid_num;
    // reference kernel_config.cuh:161-171: bucket from graph_degree once there are more than 32 centroids
    a.max_centroid = centroid_num <= 32 ? 32 : (graph_degree <= 64 ? 64 : (graph_degree <= 128 ? 128 : 256));
    if (rank_all_centroids) a.max_centroid = centroid_num <= 32 ? 32 : (centroid_num <= 64 ? 64 : (centroid_num <= 128 ? 128 : 256));
    a.top_k = top_k;
    a.query_num = query_num;
    a.p.beam = beam;
    a.p.degree = graph_degree;
    a.p.dim = dim;
    a.p.hash_bit = hash_bit;
    a.p.reset_interval = hash_reset_interval ? hash_reset_interval : 1;
    a.p.max_iterations = max_iterations;
    a.p.min_iterations = min_iterations;
    a.p.metric = metric;

    // Rows of bytes: a first launch takes the queries that are of bytes themselves and marks the others, which a second one
    // searches on the fp32 rows (on a batch without any it costs 3 us).  A batch of fractions pays for the first one: on a million rows of
    // 128 values, with it and without, 1 query at beam 32 85 : 83 us, 60 queries 112 : 109, 10 000 at beam 64 1 325 : 1 318.
    if (bytes && graph_degree <= kMostByteDegree && dim <= kMostByteDims) {
        if (reinterpret_cast<uintptr_t>(bytes) % 16) return GLIDE_ERR_BAD_ARGUMENT;
        a.bytes = bytes;
        const size_t lds_bytes = beam_lds_bytes(graph_degree) + round_up32(centroid_num) * sizeof(float) + (size_t{1} << hash_bit) * sizeof(uint32_t);
        for (const search_fn fn : {pick_search_bytes(beam, dim), pick_search_left_over(beam, dim)}) {
            GLIDE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
            hipLaunchKernelGGL(fn, dim3(query_num < kMostWorkgroups ? query_num : kMostWorkgroups), dim3(64), lds_bytes, as_stream(stream), a);
        }
        return launch_status();
    }

    const bool team = dim > 256 && static_cast<size_t>(query_num) * kTeam <= 2 * simd_count();   // see search_team_kernel
    search_fn fn = graph_degree <= 64 ? pick_search_64(beam, dim, team) : graph_degree <= 128 ? pick_search_128(beam, dim, team) : pick_search_256(beam, dim, team);
    const size_t lds_bytes = beam_lds_bytes(graph_degree) + round_up32(centroid_num) * sizeof(float) +
                             (size_t{1} << hash_bit) * sizeof(uint32_t) +
                             (team ? (dim <= 512 ? TeamShape<4>::query_bytes : dim <= 1024 ? TeamShape<8>::query_bytes : dim <= 2048 ? TeamShape<16>::query_bytes : TeamShape<32>::query_bytes) + 16 : 0);
    GLIDE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
    if (team) hipLaunchKernelGGL(fn, dim3(query_num), dim3(64 * kTeam), lds_bytes, as_stream(stream), a);
    else hipLaunchKernelGGL(fn, dim3(query_num < kMostWorkgroups ? query_num : kMostWorkgroups), dim3(64), lds_bytes, as_stream(stream), a);
    return launch_status();
}
}  // namespace

extern "C" int glide_hip_search(const float* data, uint32_t num, uint32_t dim, const uint32_t* graph, uint32_t graph_degree,
                                const float* centroids, uint32_t centroid_num, const uint32_t* start_points,
                                const float* queries, uint32_t query_num, uint32_t top_k, uint32_t beam,
                                uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                                uint32_t hash_reset_interval, int metric, uint32_t* result_ids, float* result_dists,
                                unsigned long long* counters, void* stream) {
    return launch_search(data, nullptr, num, dim, graph, graph_degree, centroids, centroid_num, false, start_points, queries, query_num, top_k, beam,
                         max_iterations, min_iterations, hash_bit, hash_reset_interval, metric, result_ids, result_dists, counters, stream);
}

extern "C" int glide_hip_search_bytes(const float* data, const void* byte_rows, uint32_t num, uint32_t dim, const uint32_t* graph,
                                      uint32_t graph_degree, const float* centroids, uint32_t centroid_num, const uint32_t* start_points,
                                      const float* queries, uint32_t query_num, uint32_t top_k, uint32_t beam, uint32_t max_iterations,
                                      uint32_t min_iterations, uint32_t hash_bit, uint32_t hash_reset_interval, int metric, uint32_t* result_ids,
                                      float* result_dists, unsigned long long* counters, void* stream) {
    return launch_search(data, static_cast<const unsigned char*>(byte_rows), num, dim, graph, graph_degree, centroids, centroid_num, false, start_points,
                         queries, query_num, top_k, beam, max_iterations, min_iterations, hash_bit, hash_reset_interval, metric, result_ids,
                         result_dists, counters, stream);
}

extern "C" int glide_hip_search_merged(const float* data, uint32_t num, uint32_t dim, const uint32_t* graph, uint32_t graph_degree,
                                       const float* centroids, uint32_t centroid_num, const uint32_t* start_points,
                                       const float* queries, uint32_t query_num, uint32_t top_k, uint32_t beam,
                                       uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                                       uint32_t hash_reset_interval, int metric, uint32_t* result_ids, float* result_dists,
                                       unsigned long long* counters, void* stream) {
    return launch_search(data, nullptr, num, dim, graph, graph_degree, centroids, centroid_num, true, start_points, queries, query_num, top_k, beam,
                         max_iterations, min_iterations, hash_bit, hash_reset_interval, metric, result_ids, result_dists, counters, stream);
}
