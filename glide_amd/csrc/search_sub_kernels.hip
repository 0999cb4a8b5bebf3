// The beam search inside one partition of the large path, for one degree bucket (GLIDE_CAND candidate slots).
// Reference: search_on_sub_kernel (search_kernel.cuh:653-765) with result_merge (:609-651).
#include "search_sub.hpp"

namespace glide {

// result_merge (search_kernel.cuh:609-651): best top_k of (running result, this partition's beam head)
template <int MAX_TOPK, int MAX_BEAM>
__device__ __forceinline__ void merge_result(const float* beam_dist, const uint32_t* beam_id, const uint32_t* map, float* final_dists,
                                             uint32_t* final_ids, uint32_t top_k, int lane) {
    constexpr int NR = WaveNet<MAX_TOPK>::NR;
    const bool live = MAX_TOPK >= 64 || lane < 32;
    float k[NR];
    uint32_t v[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const uint32_t e = NR * lane + r;
        k[r] = (live && e < top_k) ? final_dists[e] : FLT_MAX;
        v[r] = (live && e < top_k) ? final_ids[e] : kInvalid;
        const uint32_t kk = MAX_TOPK - 1 - e;
        if (live && kk < top_k) {
            const float rk = beam_dist[kk];
            if (k[r] > rk) {
                k[r] = rk;
                v[r] = map[beam_id[kk] & kClean];
            }
        }
    }
    WaveNet<MAX_TOPK>::merge(k, v, lane);
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const uint32_t e = NR * lane + r;
        if (live && e < top_k) {
            final_dists[e] = k[r];
            final_ids[e] = v[r];
        }
    }
}

// search_on_sub_kernel (search_kernel.cuh:653-765)
// Up to 64 slots on rows of up to 512 dims: five wavefronts per SIMD, for beams up to 64 five or SIX (75 registers allow it;
// which one is decided per launch, see six_resident).
// Over rows of bytes as many as the registers allow (eight up to beam 128).
// LEFT: only the pairs that the kernel for rows of bytes has left over.
constexpr int sub_waves_least(int cand, int beam, int dimv, bool six) { return dimv > 4 || dimv < 0 ? 1 : cand <= 64 ? (six ? 6 : 5) : beam > 256 ? 4 : 1; }
constexpr int sub_waves_most(int cand, int dimv, bool six) { return dimv > 4 || dimv < 0 || cand > 64 ? 8 : six ? 6 : 5; }
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool WHOLE = false, bool SIX = false, bool LEFT = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sub_waves_least(MAX_CAND, MAX_BEAM, DIMV, SIX), sub_waves_most(MAX_CAND, DIMV, SIX))))
void search_sub_kernel(SubArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    auto* lds = reinterpret_cast<BeamLds<MAX_CAND>*>(smem);
    float* head_dist = reinterpret_cast<float*>(smem + sizeof(BeamLds<MAX_CAND>));   // beam head staged for the merge (128 pairs)
    uint32_t* head_id = reinterpret_cast<uint32_t*>(head_dist + 128);
    uint32_t* hash = head_id + 128;
    uint32_t qid = blockIdx.x;
    row_data<DIMV> data;
    if constexpr (RowShape<DIMV>::BYTES) data = a.bytes;
    else data = a.data;
    const uint32_t* graph = a.graph;
    const uint32_t* map = a.map;
    uint32_t start_point = a.start_point;
    if (a.pair_segment) {
        if (qid >= a.list_len) return;
        if (LEFT && a.pair_ids[static_cast<size_t>(qid) * a.top_k] != kLeftOver) return;   // done on rows of bytes
        const uint32_t seg = a.pair_segment[qid];
        const size_t start = a.segment_starts[seg];
        data = row_at<DIMV>(data, static_cast<uint32_t>(start), a.p.dim);
        graph += start * a.p.degree;
        map += start;
        start_point = a.segment_start_points[seg];
        if (start_point == kInvalid) {   // an empty partition: nothing to find
            for (uint32_t e = lane_id(); e < a.top_k; e += 64) {
                a.pair_dists[static_cast<size_t>(blockIdx.x) * a.top_k + e] = FLT_MAX;
                a.pair_ids[static_cast<size_t>(blockIdx.x) * a.top_k + e] = kInvalid;
            }
            return;
        }
        qid = a.query_list[qid];
    } else if (a.query_list) {
        if (qid >= a.list_len) return;
        qid = a.query_list[qid];
    } else {
        if (qid >= a.query_num) return;
        bool is_search = false;   // wave-uniform scan of this query's partition list
        for (uint32_t i = 0; i < a.centroid_num; i++) {
            const uint32_t s = a.segment_ids[static_cast<size_t>(qid) * a.centroid_num + i];
            if (s == a.segment_id) { is_search = true; break; }
            if (s == kInvalid) break;
        }
        if (!is_search) return;
    }

    Beam<MAX_CAND, MAX_BEAM, DIMV, false, WHOLE> b;
    const float* query = a.queries + static_cast<size_t>(qid) * a.p.dim;
    if constexpr (RowShape<DIMV>::BYTES) {
        if (*a.other != 0 || !b.init_packing(lds, hash, a.p, query)) {   // not of bytes: left to the fp32 kernel behind this one
            if (lane_id() == 0) a.pair_ids[static_cast<size_t>(blockIdx.x) * a.top_k] = kLeftOver;
            return;
        }
    } else {
        b.init(lds, hash, a.p, query);
    }
    b.expand(start_point, graph, data, kInvalid, kInvalid);   // get_init with point_id = 0xffffffff
    b.run(graph, data, kInvalid);

    constexpr int NB = MAX_BEAM / 64;
    if (a.pair_segment) {   // the head of this pair's beam, ids already as input row numbers; merged per query afterwards
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t e = NB * b.lane + r;
            if (e < a.top_k) {
                const float d = b.bk[r];
                a.pair_dists[static_cast<size_t>(blockIdx.x) * a.top_k + e] = d;
                a.pair_ids[static_cast<size_t>(blockIdx.x) * a.top_k + e] = d < FLT_MAX ? map[b.bv[r] & kClean] : kInvalid;
            }
        }
        b.flush_counters(a.counters);
        return;
    }
#pragma unroll
    for (int r = 0; r < NB; r++) {
        const uint32_t e = NB * b.lane + r;
        if (e < 128) {
            head_dist[e] = b.bk[r];
            head_id[e] = b.bv[r];
        }
    }
    wave_sync();
    float* fd = a.final_dists + static_cast<size_t>(qid) * a.top_k;
    uint32_t* fi = a.final_ids + static_cast<size_t>(qid) * a.top_k;
    switch (a.max_topk) {   // kernel_config.cuh:312-323
        case 32: merge_result<32, MAX_BEAM>(head_dist, head_id, map, fd, fi, a.top_k, b.lane); break;
        case 64: merge_result<64, MAX_BEAM>(head_dist, head_id, map, fd, fi, a.top_k, b.lane); break;
        default: merge_result<128, MAX_BEAM>(head_dist, head_id, map, fd, fi, a.top_k, b.lane); break;
    }
    b.flush_counters(a.counters);
}

template <int MAX_CAND, int MAX_BEAM, bool WHOLE = false>
sub_fn pick_sub_dim(uint32_t dim) {
    if (dim <= 128) return search_sub_kernel<MAX_CAND, MAX_BEAM, 1, WHOLE>;
    if (dim <= 256) return search_sub_kernel<MAX_CAND, MAX_BEAM, 2, WHOLE>;
    if (dim <= 512) return search_sub_kernel<MAX_CAND, MAX_BEAM, 4, WHOLE>;
    if (dim <= 1024) return search_sub_kernel<MAX_CAND, MAX_BEAM, 8, WHOLE>;
    if (dim <= 2048) return search_sub_kernel<MAX_CAND, MAX_BEAM, 16, WHOLE>;
    return search_sub_kernel<MAX_CAND, MAX_BEAM, 32, WHOLE>;
}
template <int MAX_CAND>
sub_fn pick_sub_beam(uint32_t beam, uint32_t dim, bool six) {
    if constexpr (MAX_CAND <= 64) {
        if (beam <= 64 && dim <= 512 && six) return dim <= 128 ? search_sub_kernel<MAX_CAND, 64, 1, false, true> : dim <= 256 ? search_sub_kernel<MAX_CAND, 64, 2, false, true> : search_sub_kernel<MAX_CAND, 64, 4, false, true>;
    }
    if (beam <= 64) return pick_sub_dim<MAX_CAND, 64>(dim);
    if (beam <= 128) return pick_sub_dim<MAX_CAND, 128>(dim);
    if (beam <= 256) return pick_sub_dim<MAX_CAND, 256>(dim);
    if (beam == 512) return pick_sub_dim<MAX_CAND, 512, true>(dim);   // the whole of the widest beam: merged in the registers
    return pick_sub_dim<MAX_CAND, 512>(dim);
}

#if GLIDE_CAND == 64
template <int DIMV, bool LEFT>
sub_fn pick_sub_bytes_beam(uint32_t beam) {
    if (beam <= 64) return search_sub_kernel<64, 64, DIMV, false, false, LEFT>;
    if (beam <= 128) return search_sub_kernel<64, 128, DIMV, false, false, LEFT>;
    if (beam <= 256) return search_sub_kernel<64, 256, DIMV, false, false, LEFT>;
    if (beam == 512) return search_sub_kernel<64, 512, DIMV, true, false, LEFT>;
    return search_sub_kernel<64, 512, DIMV, false, false, LEFT>;
}
sub_fn pick_sub_bytes(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_sub_bytes_beam<-1, false>(beam) : pick_sub_bytes_beam<-2, false>(beam); }
sub_fn pick_sub_left_over(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_sub_bytes_beam<1, true>(beam) : pick_sub_bytes_beam<2, true>(beam); }
#endif

#define GLIDE_PICK_NAME(cand) pick_sub_##cand
#define GLIDE_PICK(cand) GLIDE_PICK_NAME(cand)
sub_fn GLIDE_PICK(GLIDE_CAND)(uint32_t beam, uint32_t dim, bool six) { return pick_sub_beam<GLIDE_CAND>(beam, dim, six); }

}  // namespace glide
