// One query per wavefront beam search over the finished index, for one degree bucket (GLIDE_CAND candidate slots).
// Reference: search_kernel (search_kernel.cuh:393-490) launched by GLIDE::search (glide_impl.cuh:370-454).
#include "search.hpp"

namespace glide {

template <int DIMV, bool TEAM = false>
__device__ __forceinline__ uint32_t pick_centroid(uint32_t max_centroid, const RowRegs<DIMV>& q, const float* centroids,
                                                  uint32_t centroid_num, uint32_t dim, int metric, float* scratch, int lane) {
    switch (max_centroid) {  // bucket chosen like reference kernel_config.cuh:161-171
        case 32: return nearest_centroid<32, DIMV, TEAM>(q, centroids, centroid_num, dim, metric, scratch, lane);
        case 64: return nearest_centroid<64, DIMV, TEAM>(q, centroids, centroid_num, dim, metric, scratch, lane);
        case 128: return nearest_centroid<128, DIMV, TEAM>(q, centroids, centroid_num, dim, metric, scratch, lane);
        default: return nearest_centroid<256, DIMV, TEAM>(q, centroids, centroid_num, dim, metric, scratch, lane);
    }
}

// LEFT: only the queries that the kernel for rows of bytes has left over.
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool WHOLE, bool LEFT>
__device__ __forceinline__ void search_body(const SearchArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    auto* lds = reinterpret_cast<BeamLds<MAX_CAND>*>(smem);
    uint32_t* hash = reinterpret_cast<uint32_t*>(smem + sizeof(BeamLds<MAX_CAND>));   // at a constant offset: no addition a probe
    float* cent = reinterpret_cast<float*>(hash + (1u << a.p.hash_bit));
    // one query a workgroup, as far as a launch has workgroups
    for (uint32_t qid = blockIdx.x; qid < a.query_num; qid += gridDim.x) {
        Beam<MAX_CAND, MAX_BEAM, DIMV, false, WHOLE> b;
        const float* query = a.queries + static_cast<size_t>(qid) * a.p.dim;
        row_data<DIMV> rows;
        uint32_t c0;
        if constexpr (RowShape<DIMV>::BYTES) {
            constexpr int F = -DIMV;   // centroids are fp32: the shape of an fp32 row of this length
            if (!b.init_packing(lds, hash, a.p, query)) {   // not of bytes: left to the fp32 kernel behind this one
                if (b.lane == 0) a.result_ids[static_cast<size_t>(qid) * a.top_k] = kLeftOver;
                continue;
            }
            rows = a.bytes;
            RowRegs<F> q;
            load_row<F>(q, query, a.p.dim, RowShape<F>::lane_in_row(b.lane));
            c0 = pick_centroid<F>(a.max_centroid, q, a.centroids, a.centroid_num, a.p.dim, a.p.metric, cent, b.lane);
        } else {
            if (LEFT && a.result_ids[static_cast<size_t>(qid) * a.top_k] != kLeftOver) continue;   // done on rows of bytes
            b.init(lds, hash, a.p, query);
            rows = a.data;
            c0 = pick_centroid<DIMV>(a.max_centroid, b.q, a.centroids, a.centroid_num, a.p.dim, a.p.metric, cent, b.lane);
        }
        const uint32_t entry = a.start_points[c0];
        b.expand(entry, a.graph, rows, kInvalid, kInvalid);  // result_init: entry node itself is never scored
        b.run(a.graph, rows, kInvalid);

        constexpr int NB = MAX_BEAM / 64;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t e = NB * b.lane + r;
            if (e < a.top_k) {
                a.result_ids[static_cast<size_t>(qid) * a.top_k + e] = b.bv[r] & kClean;
                a.result_dists[static_cast<size_t>(qid) * a.top_k + e] = b.bk[r];
            }
        }
        b.flush_counters(a.counters);
        wave_sync();   // the next query reuses the LDS
    }
}

// Rows of up to 512 dims and up to 64 slots: six wavefronts per SIMD (80 registers; beams up to 128 need no more anyway,
// beam 256 would take 84), above beam 256 five (96 of 97).  These searches wait for their gathers and their own dependent
// steps, and a wavefront more is worth it.  Wider buckets hold several slots a lane and keep the bounds they were measured at.
template <int MAX_CAND, int MAX_BEAM, int DIMV>
constexpr int search_waves() {
    if (DIMV > 4) return 1;
    if (MAX_CAND <= 64) return MAX_BEAM > 256 ? 5 : 6;
    return MAX_BEAM > 256 ? 4 : MAX_BEAM == 256 && MAX_CAND <= 128 ? 5 : 1;
}
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool WHOLE = false, bool LEFT = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(search_waves<MAX_CAND, MAX_BEAM, DIMV>())))
void search_kernel(SearchArgs a) {
    search_body<MAX_CAND, MAX_BEAM, DIMV, WHOLE, LEFT>(a);
}

// Small batches of long rows (more than 256 dims): a team of kTeam wavefronts per query.  Wavefront 0 owns the search
// (beam, visited set, sorting networks) exactly as in search_kernel; between two of its passes every wavefront of the
// team scores a share of the expansion's candidate rows.  One wavefront can keep only a few 2-4 KB rows in flight in its
// registers, and a search is a chain of dependent expansions: while the batch leaves SIMDs idle, a team gives a query
// kTeam times the bytes on their way and an expansion takes one or two memory round trips instead of six (64 queries of
// 960 dims: 1.9 times the throughput at beams up to 256, 1.3 times above).  Once a batch fills the chip on its own
// (about two wavefronts per SIMD) the row gathers run at the rate the memory system sustains for scattered rows either
// way and the team only adds its barriers, so larger batches keep one wavefront per query.  The query row sits in LDS
// once per team (RefInLds) so that the registers hold rows in flight; every distance is summed in the order
// search_kernel sums it, so results are identical.
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool WHOLE = false>
__global__ __launch_bounds__(64 * kTeam) void search_team_kernel(SearchArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    using Shape = RowShape<DIMV>;
    auto* lds = reinterpret_cast<BeamLds<MAX_CAND>*>(smem);
    float4* qlds = reinterpret_cast<float4*>(smem + sizeof(BeamLds<MAX_CAND>));
    uint32_t* ctl = reinterpret_cast<uint32_t*>(qlds + Shape::NV * Shape::LPR);   // [0] rows to score, [1] search over
    uint32_t* hash = ctl + 4;
    float* cent = reinterpret_cast<float*>(hash + (1u << a.p.hash_bit));
    const uint32_t wave = threadIdx.x >> 6;
    const int lane = lane_id();
    for (uint32_t qid = blockIdx.x; qid < a.query_num; qid += gridDim.x) {
        Beam<MAX_CAND, MAX_BEAM, DIMV, true, WHOLE> b;
        uint32_t iter = 0;
        bool terminate = false;
        if (wave == 0) {
            b.init(lds, hash, a.p, a.queries + static_cast<size_t>(qid) * a.p.dim);
            if (Shape::row_of_lane(lane) == 0) {
#pragma unroll
                for (int c = 0; c < Shape::NV; c++) qlds[c * Shape::LPR + Shape::lane_in_row(lane)] = b.q.v[c];
            }
            const uint32_t c0 = pick_centroid<DIMV, true>(a.max_centroid, b.q, a.centroids, a.centroid_num, a.p.dim, a.p.metric, cent, lane);
            const uint32_t nv = b.expand_list(a.start_points[c0], a.graph, kInvalid, kInvalid);   // result_init: the entry node itself is never scored
            if (lane == 0) {
                ctl[0] = nv;
                ctl[1] = 0;
            }
        }
        __syncthreads();
        while (true) {
            const uint32_t nv = ctl[0];
            score_share<DIMV, TeamShape<DIMV>::U>(RefInLds<DIMV>{qlds}, a.data, a.p.dim, 0, nv, lane, wave, kTeam,
                                                  [lds](uint32_t idx) { return lds->vlist[idx]; },
                                                  [lds](uint32_t idx, float sq) { lds->cand_dist[idx] = sq; });
            __syncthreads();
            if (wave == 0) {
                uint32_t next = 0;
                const bool more = b.step_to_list(iter, terminate, a.graph, kInvalid, next);
                if (lane == 0) {
                    ctl[0] = next;
                    ctl[1] = more ? 0u : 1u;
                }
            }
            __syncthreads();
            if (ctl[1] != 0) break;
        }
        if (wave == 0) {
            constexpr int NB = MAX_BEAM / 64;
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const uint32_t e = NB * lane + r;
                if (e < a.top_k) {
                    a.result_ids[static_cast<size_t>(qid) * a.top_k + e] = b.bv[r] & kClean;
                    a.result_dists[static_cast<size_t>(qid) * a.top_k + e] = b.bk[r];
                }
            }
            b.flush_counters(a.counters);
        }
        __syncthreads();   // the next query reuses the LDS
    }
}

template <int MAX_CAND, int MAX_BEAM, bool WHOLE = false>
search_fn pick_dim(uint32_t dim) {
    if (dim <= 128) return search_kernel<MAX_CAND, MAX_BEAM, 1, WHOLE>;
    if (dim <= 256) return search_kernel<MAX_CAND, MAX_BEAM, 2, WHOLE>;
    if (dim <= 512) return search_kernel<MAX_CAND, MAX_BEAM, 4, WHOLE>;
    if (dim <= 1024) return search_kernel<MAX_CAND, MAX_BEAM, 8, WHOLE>;
    if (dim <= 2048) return search_kernel<MAX_CAND, MAX_BEAM, 16, WHOLE>;
    return search_kernel<MAX_CAND, MAX_BEAM, 32, WHOLE>;
}
template <int MAX_CAND, int MAX_BEAM, bool WHOLE = false>
search_fn pick_team_dim(uint32_t dim) {
    if (dim <= 512) return search_team_kernel<MAX_CAND, MAX_BEAM, 4, WHOLE>;
    if (dim <= 1024) return search_team_kernel<MAX_CAND, MAX_BEAM, 8, WHOLE>;
    if (dim <= 2048) return search_team_kernel<MAX_CAND, MAX_BEAM, 16, WHOLE>;
    return search_team_kernel<MAX_CAND, MAX_BEAM, 32, WHOLE>;
}
template <int MAX_CAND>
search_fn pick_team_beam(uint32_t beam, uint32_t dim) {
    if (beam <= 64) return pick_team_dim<MAX_CAND, 64>(dim);
    if (beam <= 128) return pick_team_dim<MAX_CAND, 128>(dim);
    if (beam <= 256) return pick_team_dim<MAX_CAND, 256>(dim);
    if (beam == 512) return pick_team_dim<MAX_CAND, 512, true>(dim);
    return pick_team_dim<MAX_CAND, 512>(dim);
}
template <int MAX_CAND>
search_fn pick_beam(uint32_t beam, uint32_t dim) {
    if (beam <= 64) return pick_dim<MAX_CAND, 64>(dim);
    if (beam <= 128) return pick_dim<MAX_CAND, 128>(dim);
    if (beam <= 256) return pick_dim<MAX_CAND, 256>(dim);
    if (beam == 512) return pick_dim<MAX_CAND, 512, true>(dim);
    return pick_dim<MAX_CAND, 512>(dim);
}

#if GLIDE_CAND == 64
template <int DIMV, bool LEFT = false>
search_fn pick_bytes_beam(uint32_t beam) {
    if (beam <= 64) return search_kernel<64, 64, DIMV, false, LEFT>;
    if (beam <= 128) return search_kernel<64, 128, DIMV, false, LEFT>;
    if (beam <= 256) return search_kernel<64, 256, DIMV, false, LEFT>;
    if (beam == 512) return search_kernel<64, 512, DIMV, true, LEFT>;
    return search_kernel<64, 512, DIMV, false, LEFT>;
}
search_fn pick_search_bytes(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_bytes_beam<-1>(beam) : pick_bytes_beam<-2>(beam); }
search_fn pick_search_left_over(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_bytes_beam<1, true>(beam) : pick_bytes_beam<2, true>(beam); }
#endif

#define GLIDE_PICK_NAME(cand) pick_search_##cand
#define GLIDE_PICK(cand) GLIDE_PICK_NAME(cand)
search_fn GLIDE_PICK(GLIDE_CAND)(uint32_t beam, uint32_t dim, bool team) {
    return team ? pick_team_beam<GLIDE_CAND>(beam, dim) : pick_beam<GLIDE_CAND>(beam, dim);
}

}  // namespace glide
