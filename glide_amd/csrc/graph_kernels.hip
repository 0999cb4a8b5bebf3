// Sub-graph build with pruning and refinement, one point per wavefront, for one degree bucket (GLIDE_CAND candidate slots).
// Reference: graph_kernel.cuh (build_kernel :249-316, build_boundary_kernel :318-376, refine_kernel :580-673).
#include "graph.hpp"

namespace glide {

// Up to 64 slots on rows of up to 512 dims, here and in refine_kernel: six wavefronts per SIMD (80 registers; beams up to
// 128 need no more anyway, beam 256 would take up to 84), five above beam 256 (96) and where rows are looked at in fp16 first
// (32 rows of them on their way; with six and 16 rows 250 000 rows of 128 values build in 77 ms instead of 59).
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool ROUGH = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(DIMV > 4 || MAX_CAND > 64 ? 1 : MAX_BEAM > 256 || ROUGH ? 5 : 6))) void build_kernel(BuildArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    auto* lds = reinterpret_cast<BeamLds<MAX_CAND>*>(smem);
    auto* pl = reinterpret_cast<PruneLds<MAX_BEAM>*>(smem + sizeof(BeamLds<MAX_CAND>));
    uint32_t* hash = reinterpret_cast<uint32_t*>(smem + sizeof(BeamLds<MAX_CAND>) + sizeof(PruneLds<MAX_BEAM>));
    if (blockIdx.x >= a.point_count) return;
    const uint32_t point = a.first_point + blockIdx.x;
    const bool boundary = a.boundary_start != kInvalid;

    const bool segment_mode = a.map == nullptr;   // one staged partition: local ids in and out (build_for_large_kernel)
    uint32_t seg_start, entry;
    if (segment_mode) {
        seg_start = 0;
        entry = a.boundary_start_point;
    } else if (boundary) {
        seg_start = a.boundary_start;
        entry = a.boundary_start_point;
    } else {
        uint32_t seg = 0;
        for (; seg < a.segment_num; seg++)
            if (point < a.segment_starts[seg] + a.segment_lengths[seg]) break;
        seg_start = a.segment_starts[seg];
        entry = a.start_points[seg];
    }
    row_data<DIMV> rows;
    if constexpr (RowShape<DIMV>::BYTES) rows = a.bytes;
    else rows = a.reorder_data;
    const row_data<DIMV> sdata = row_at<DIMV>(rows, seg_start, a.p.dim);
    const uint32_t* sgraph = a.knn_graph + static_cast<size_t>(seg_start) * a.p.degree;

    Beam<MAX_CAND, MAX_BEAM, DIMV, false, false, ROUGH> b;
    b.init(lds, hash, a.p, row_at<DIMV>(rows, point, a.p.dim));
    RoughPool look{};
    if constexpr (ROUGH) {
        static_assert(sizeof(lds->pool_open) / 4 >= MAX_BEAM, "room for every entry of a pool");
        look = RoughPool{rough_rows(a.rough, a.p.dim), lds->pool_open};
        b.look_first(look.rough, point, seg_start);
    }
    // get_init (search_kernel.cuh:336-360): all neighbours of the entry are hashed; the one whose *local* id equals
    // this point's *reorder* id is left unscored (the reference compares across id spaces, graph_kernel.cuh:295-298)
    b.expand(entry, sgraph, sdata, kInvalid, point);
    b.run(sgraph, sdata, point - seg_start);

    uint32_t pool = beam_to_pool(b, pl);
    prune_pool<MAX_BEAM, DIMV, ROUGH>(pl, look, pool, rows, a.p.dim, seg_start, a.graph_degree, a.relaxant, a.p.metric, b.lane,
                               b.cnt.rows_scored);
    wave_sync();
    if (segment_mode) {   // map_to_graph (graph_kernel.cuh:145-150)
        uint32_t* row = a.graph + static_cast<size_t>(point) * a.graph_degree;
        for (uint32_t i = b.lane; i < a.graph_degree; i += 64) row[i] = pl->neighbor[i];
        b.flush_counters(a.counters);
        return;
    }
    uint32_t* row = a.graph + static_cast<size_t>(a.map[point]) * a.graph_degree;
    if (boundary) {
        merge_boundary_row<MAX_BEAM>(pl, row, a.map, a.graph_degree, b.lane);
    } else {  // map_to_graph_sub (graph_kernel.cuh:152-158)
        for (uint32_t i = b.lane; i < a.graph_degree; i += 64) {
            const uint32_t nb = pl->neighbor[i];
            row[i] = nb == kInvalid ? kInvalid : a.map[nb];
        }
    }
    b.flush_counters(a.counters);
}

template <int DIMV>
__device__ __forceinline__ uint32_t pick_centroid_refine(uint32_t max_centroid, const RowRegs<DIMV>& q, const float* centroids,
                                                         uint32_t centroid_num, uint32_t dim, int metric, float* scratch, int lane) {
    switch (max_centroid) {
        case 32: return nearest_centroid<32, DIMV>(q, centroids, centroid_num, dim, metric, scratch, lane);
        case 64: return nearest_centroid<64, DIMV>(q, centroids, centroid_num, dim, metric, scratch, lane);
        case 128: return nearest_centroid<128, DIMV>(q, centroids, centroid_num, dim, metric, scratch, lane);
        default: return nearest_centroid<256, DIMV>(q, centroids, centroid_num, dim, metric, scratch, lane);
    }
}

// Rows are read from graph_in and written to graph_out (every row is written: copied, with its empty slots
// filled).  The reference refines in place while other blocks still traverse the rows.
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool ROUGH = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(DIMV > 4 || MAX_CAND > 64 ? 1 : MAX_BEAM > 256 || ROUGH ? 5 : 6))) void refine_kernel(RefineArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    auto* lds = reinterpret_cast<BeamLds<MAX_CAND>*>(smem);
    using Prune = PruneLds<MAX_BEAM, (MAX_CAND < 64 ? 64 : MAX_CAND)>;   // the row has at most MAX_CAND slots here
    auto* pl = reinterpret_cast<Prune*>(smem + sizeof(BeamLds<MAX_CAND>));
    uint32_t* hash = reinterpret_cast<uint32_t*>(smem + sizeof(BeamLds<MAX_CAND>) + sizeof(Prune));   // at a constant offset: no addition a probe
    float* cent = reinterpret_cast<float*>(hash + (1u << a.p.hash_bit));
    if (blockIdx.x >= a.num) return;
    const uint32_t point = a.order ? a.order[blockIdx.x] : blockIdx.x;
    if (point >= a.num) return;
    const int lane = lane_id();
    const uint32_t D = a.p.degree;
    const uint32_t* in_row = a.graph_in + static_cast<size_t>(point) * D;
    uint32_t* out_row = a.graph_out + static_cast<size_t>(point) * D;

    uint32_t need = 0;
    for (uint32_t base = 0; base < Prune::kCap; base += 64) {
        const uint32_t i = base + lane;
        const uint32_t g = i < D ? in_row[i] : kInvalid;
        pl->s_graph[i] = g;
        if (i < D) out_row[i] = g;
        need += __popcll(ballot(i < D && g == kInvalid));
    }
    wave_sync();
    if (need == 0) return;

    Beam<MAX_CAND, MAX_BEAM, DIMV, false, false, ROUGH> b;
    row_data<DIMV> rows;
    if constexpr (RowShape<DIMV>::BYTES) rows = a.bytes;
    else rows = a.data;
    b.init(lds, hash, a.p, row_at<DIMV>(rows, point, a.p.dim));
    RoughPool look{};
    if constexpr (ROUGH) {
        static_assert(sizeof(lds->pool_open) / 4 >= MAX_BEAM, "room for every entry of a pool");
        look = RoughPool{rough_rows(a.rough, a.p.dim), lds->pool_open};
        b.look_first(look.rough, point, 0u);
    }
    if (a.centroids != nullptr) {
        uint32_t c0;
        if constexpr (RowShape<DIMV>::BYTES) {
            constexpr int F = -DIMV;   // centroids are fp32: the shape of an fp32 row of this length
            RowRegs<F> q;
            load_row<F>(q, a.data + static_cast<size_t>(point) * a.p.dim, a.p.dim, RowShape<F>::lane_in_row(lane));
            c0 = pick_centroid_refine<F>(a.max_centroid, q, a.centroids, a.centroid_num, a.p.dim, a.p.metric, cent, lane);
        } else {
            c0 = pick_centroid_refine<DIMV>(a.max_centroid, b.q, a.centroids, a.centroid_num, a.p.dim, a.p.metric, cent, lane);
        }
        b.expand(a.start_points[c0], a.graph_in, rows, kInvalid, kInvalid);
    } else {   // refine_for_large_kernel (graph_kernel.cuh:796-798): get_init from the segment's start point
        b.expand(a.segment_start_point, a.graph_in, rows, kInvalid, point);
    }
    b.run(a.graph_in, rows, point);

    uint32_t pool = beam_to_pool(b, pl);
    prune_pool_refine<MAX_BEAM, DIMV, ROUGH>(pl, look, pool, rows, a.p.dim, point, D, need, a.relaxant, a.p.metric, lane, b.cnt.rows_scored);
    wave_sync();
    uint32_t used = 0;
    for (uint32_t base = 0; base < round_up32(D); base += 64) {  // holes in slot order (graph_kernel.cuh:659-671)
        const uint32_t i = base + lane;
        const bool hole = i < D && pl->s_graph[i] == kInvalid;
        const uint64_t m = ballot(hole);
        if (hole) out_row[i] = pl->neighbor[used + prefix_count(m)];
        used += __popcll(m);
    }
    b.flush_counters(a.counters);
}

template <int MAX_CAND, int MAX_BEAM>
build_fn pick_build_dim(uint32_t dim) {
    if (dim <= 128) return build_kernel<MAX_CAND, MAX_BEAM, 1>;
    if (dim <= 256) return build_kernel<MAX_CAND, MAX_BEAM, 2>;
    if (dim <= 512) return build_kernel<MAX_CAND, MAX_BEAM, 4>;
    if (dim <= 1024) return build_kernel<MAX_CAND, MAX_BEAM, 8>;
    if (dim <= 2048) return build_kernel<MAX_CAND, MAX_BEAM, 16>;
    return build_kernel<MAX_CAND, MAX_BEAM, 32>;
}
template <int MAX_CAND>
build_fn pick_build_beam(uint32_t beam, uint32_t dim) {
    if (beam <= 64) return pick_build_dim<MAX_CAND, 64>(dim);
    if (beam <= 128) return pick_build_dim<MAX_CAND, 128>(dim);
    if (beam <= 256) return pick_build_dim<MAX_CAND, 256>(dim);
    return pick_build_dim<MAX_CAND, 512>(dim);
}
template <int MAX_CAND, int MAX_BEAM>
refine_fn pick_refine_dim(uint32_t dim) {
    if (dim <= 128) return refine_kernel<MAX_CAND, MAX_BEAM, 1>;
    if (dim <= 256) return refine_kernel<MAX_CAND, MAX_BEAM, 2>;
    if (dim <= 512) return refine_kernel<MAX_CAND, MAX_BEAM, 4>;
    if (dim <= 1024) return refine_kernel<MAX_CAND, MAX_BEAM, 8>;
    if (dim <= 2048) return refine_kernel<MAX_CAND, MAX_BEAM, 16>;
    return refine_kernel<MAX_CAND, MAX_BEAM, 32>;
}
template <int MAX_CAND>
refine_fn pick_refine_beam(uint32_t beam, uint32_t dim) {
    if (beam <= 64) return pick_refine_dim<MAX_CAND, 64>(dim);
    if (beam <= 128) return pick_refine_dim<MAX_CAND, 128>(dim);
    if (beam <= 256) return pick_refine_dim<MAX_CAND, 256>(dim);
    return pick_refine_dim<MAX_CAND, 512>(dim);
}

#if GLIDE_CAND == 64
template <int DIMV>
build_fn pick_build_bytes_beam(uint32_t beam) {
    if (beam <= 64) return build_kernel<64, 64, DIMV>;
    if (beam <= 128) return build_kernel<64, 128, DIMV>;
    if (beam <= 256) return build_kernel<64, 256, DIMV>;
    return build_kernel<64, 512, DIMV>;
}
template <int DIMV>
refine_fn pick_refine_bytes_beam(uint32_t beam) {
    if (beam <= 64) return refine_kernel<64, 64, DIMV>;
    if (beam <= 128) return refine_kernel<64, 128, DIMV>;
    if (beam <= 256) return refine_kernel<64, 256, DIMV>;
    return refine_kernel<64, 512, DIMV>;
}
build_fn pick_build_bytes(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_build_bytes_beam<-1>(beam) : pick_build_bytes_beam<-2>(beam); }
template <int DIMV> build_fn pick_build_rough_dimv(uint32_t beam) { return beam <= 64 ? build_kernel<64, 64, DIMV, true> : build_kernel<64, 128, DIMV, true>; }
template <int DIMV> refine_fn pick_refine_rough_dimv(uint32_t beam) { return beam <= 64 ? refine_kernel<64, 64, DIMV, true> : refine_kernel<64, 128, DIMV, true>; }
build_fn pick_build_rough(uint32_t beam, uint32_t dim) {
    return dim <= 128 ? pick_build_rough_dimv<1>(beam) : dim <= 256 ? pick_build_rough_dimv<2>(beam) : dim <= 512 ? pick_build_rough_dimv<4>(beam) : pick_build_rough_dimv<8>(beam);
}
refine_fn pick_refine_rough(uint32_t beam, uint32_t dim) {
    return dim <= 128 ? pick_refine_rough_dimv<1>(beam) : dim <= 256 ? pick_refine_rough_dimv<2>(beam) : dim <= 512 ? pick_refine_rough_dimv<4>(beam) : pick_refine_rough_dimv<8>(beam);
}
refine_fn pick_refine_bytes(uint32_t beam, uint32_t dim) { return dim <= 128 ? pick_refine_bytes_beam<-1>(beam) : pick_refine_bytes_beam<-2>(beam); }
#endif

#define GLIDE_PICK_NAME(kind, cand) pick_##kind##_##cand
#define GLIDE_PICK(kind, cand) GLIDE_PICK_NAME(kind, cand)
build_fn GLIDE_PICK(build, GLIDE_CAND)(uint32_t beam, uint32_t dim) { return pick_build_beam<GLIDE_CAND>(beam, dim); }
refine_fn GLIDE_PICK(refine, GLIDE_CAND)(uint32_t beam, uint32_t dim) { return pick_refine_beam<GLIDE_CAND>(beam, dim); }

}  // namespace glide
