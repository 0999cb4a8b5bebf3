// Graph construction kernels: per-partition sub-graph build with pruning, cross-partition (boundary) merge,
// reverse-edge insertion and refinement.  One point per wavefront.
// Reference: graph_kernel.cuh (build_kernel :249-316, build_boundary_kernel :318-376, reverse_graph_kernel
// :378-414, insert_reverse_kernel :416-453, refine_kernel :580-673) as sequenced by glide_impl.cuh:77-316.
#include "graph.hpp"
#include "host_util.hpp"

namespace glide {

// ------------------------------------------------------------------------------------------ reverse edges
// Reference order of arrival in a row's reverse list is whatever the atomics give; here the list is the D
// smallest (column, source) pairs, i.e. the order of a sequential sweep over columns then sources.
//
// pass 1: one wavefront per source s.  For each column c with target t = graph[s][c] < num, the row of t is read
// coalesced and searched for s.  Missing pairs are counted per target and remembered in a bit per (s, c).
__global__ __launch_bounds__(256) void reverse_count_kernel(const uint32_t* graph, uint32_t num, uint32_t D, uint32_t* miss_bits,
                                                            uint32_t* counts) {
    const int lane = lane_id();
    const uint32_t s = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (s >= num) return;
    const uint32_t words = ceil_div(D, 32);
    for (uint32_t cb = 0; cb < D; cb += 32) {
        uint32_t bits = 0;
        const uint32_t cend = cb + 32 < D ? cb + 32 : D;
        for (uint32_t c = cb; c < cend; c++) {
            const uint32_t t = graph[static_cast<size_t>(s) * D + c];   // wave-uniform
            if (t >= num) continue;
            bool have = false;
            for (uint32_t i = lane; i < D; i += 64) have |= graph[static_cast<size_t>(t) * D + i] == s;
            if (ballot(have) == 0) {
                bits |= 1u << (c - cb);
                if (lane == 0) atomicAdd(&counts[t], 1u);
            }
        }
        if (lane == 0) miss_bits[static_cast<size_t>(s) * words + cb / 32] = bits;
    }
}

// pass 2: bucket offsets (any order; only the bucket contents matter)
__global__ void reverse_offsets_kernel(const uint32_t* counts, uint32_t num, uint32_t* offsets, unsigned long long* cursor) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= num) return;
    const uint32_t c = counts[t];
    offsets[t] = c ? static_cast<uint32_t>(atomicAdd(cursor, static_cast<unsigned long long>(c))) : 0u;
}

// pass 3: scatter (column, source) keys into the target's bucket
__global__ void reverse_scatter_kernel(const uint32_t* graph, uint32_t num, uint32_t D, const uint32_t* miss_bits,
                                       const uint32_t* offsets, uint32_t* fill, unsigned long long* pool) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= num) return;
    const uint32_t words = ceil_div(D, 32);
    for (uint32_t w = 0; w < words; w++) {
        uint32_t bits = miss_bits[static_cast<size_t>(s) * words + w];
        while (bits) {
            const uint32_t c = w * 32 + __builtin_ctz(bits);
            bits &= bits - 1;
            const uint32_t t = graph[static_cast<size_t>(s) * D + c];
            const uint32_t pos = atomicAdd(&fill[t], 1u);
            pool[static_cast<size_t>(offsets[t]) + pos] = (static_cast<unsigned long long>(c) << 32) | s;
        }
    }
}

// pass 4: one wavefront per target: the min(count, D) smallest keys of its bucket, ascending -> reverse list
__global__ __launch_bounds__(256) void reverse_select_kernel(uint32_t num, uint32_t D, const uint32_t* counts, const uint32_t* offsets,
                                                             const unsigned long long* pool, uint32_t* reverse_graph) {
    const int lane = lane_id();
    const uint32_t t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= num) return;
    const uint32_t cnt = counts[t];
    const uint32_t take = cnt < D ? cnt : D;
    const unsigned long long* bucket = pool + offsets[t];
    unsigned long long last = 0;
    bool have_last = false;
    for (uint32_t k = 0; k < take; k++) {
        unsigned long long best = ~0ull;
        for (uint32_t i = lane; i < cnt; i += 64) {
            const unsigned long long key = bucket[i];
            if ((!have_last || key > last) && key < best) best = key;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const unsigned long long o = __shfl_xor(best, off);
            best = o < best ? o : best;
        }
        last = best;
        have_last = true;
        if (lane == 0) reverse_graph[static_cast<size_t>(t) * D + k] = static_cast<uint32_t>(best & 0xffffffffull);
    }
    for (uint32_t k = take + lane; k < D; k += 64) reverse_graph[static_cast<size_t>(t) * D + k] = kInvalid;
}

// insert_reverse_kernel (graph_kernel.cuh:416-453): empty slots, in order, take the first reverse edges
__global__ __launch_bounds__(256) void insert_reverse_kernel(uint32_t* graph, const uint32_t* reverse_graph, const uint32_t* counts,
                                                             uint32_t num, uint32_t D) {
    const int lane = lane_id();
    const uint32_t p = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (p >= num) return;
    const uint32_t nrev = counts[p] > D ? D : counts[p];
    uint32_t used = 0;
    for (uint32_t base = 0; base < D && used < nrev; base += 64) {
        const uint32_t i = base + lane;
        const bool hole = i < D && graph[static_cast<size_t>(p) * D + i] == kInvalid;
        const uint64_t m = ballot(hole);
        const uint32_t pos = used + prefix_count(m);
        if (hole && pos < nrev) graph[static_cast<size_t>(p) * D + i] = reverse_graph[static_cast<size_t>(p) * D + pos];
        used += __popcll(m);
    }
}

// ------------------------------------------------------------------------------------------ rows as bytes
// fp32 rows -> bytes, zeros behind them, sixteen dims a thread; *other is set if a value is no whole number 0 .. 255.  Bound by
// reading the rows (1M x 128: 0.11 ms, 5.9 TB/s with what it writes).  The first workgroups are a launch of their own: rows
// of fractions end there, and the others find the word set and leave (in one launch every wavefront reads its rows before
// the word says anything, and all of them write it: 0.36 ms for 300k x 96 fractions).
constexpr uint32_t kPackProbe = 64;
constexpr size_t kMostPacked = size_t{16} << 32;   // bytes written at most: 2^32 threads (2^29 rows of up to 128 dims)
__global__ __launch_bounds__(256) void pack_bytes_kernel(const float* rows, uint32_t num, uint32_t dim, uint32_t lanes, uint32_t first_block, uint4* bytes,
                                                         uint32_t* other) {
    if (*other != 0) return;
    const size_t i = static_cast<size_t>(first_block + blockIdx.x) * 256 + threadIdx.x;
    const size_t row = i / lanes;
    bool exact = true;
    if (row < num) {
        uint4 out;
        exact = pack_bytes(rows + row * dim, 16 * static_cast<uint32_t>(i % lanes), dim, out);
        bytes[i] = out;
    }
    if (ballot(!exact) != 0 && lane_id() == 0) *other = 1u;
}

// ------------------------------------------------------------------------------------------ rows in fp16
// The largest |value| as bits (what is no number orders last), then every value times the power of two that it fixes.
__global__ __launch_bounds__(256) void rough_range_kernel(const float* rows, size_t quads, uint32_t* max_bits) {
    uint32_t m = 0;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < quads; i += static_cast<size_t>(gridDim.x) * 256) {
        const uint4 q = reinterpret_cast<const uint4*>(rows)[i];
        const uint32_t v[4] = {q.x & kClean, q.y & kClean, q.z & kClean, q.w & kClean};
#pragma unroll
        for (int e = 0; e < 4; e++) m = v[e] > m ? v[e] : m;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), off));
        m = o > m ? o : m;
    }
    __shared__ uint32_t of_wave[4];
    if (lane_id() == 0) of_wave[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < 4; w++) m = of_wave[w] > m ? of_wave[w] : m;
        if (m) atomicMax(max_bits, m);
    }
}
// Sixteen lanes a row.
__global__ __launch_bounds__(256) void rough_pack_kernel(const float* rows, uint32_t num, uint32_t dim, const uint32_t* max_bits, uint32_t* turn_bits,
                                                         _Float16* out) {
    const float unit = rough_unit(*max_bits), scale = 1.f / unit;   // powers of two: exact
    const float t = sqrtf(static_cast<float>(dim)) * 6.2e-5f * unit;
    const uint32_t stride = rough_stride(dim), lane = threadIdx.x % 16;
    float most = 0.f;
    for (size_t row = static_cast<size_t>(blockIdx.x) * 16 + threadIdx.x / 16; row < num; row += static_cast<size_t>(gridDim.x) * 16) {
        float off = 0.f, length = 0.f;
        for (uint32_t d0 = lane * 8; d0 < stride; d0 += 128) {
            const float* from = rows + row * dim + d0;
            const float4 x = *reinterpret_cast<const float4*>(from);
            const float4 y = d0 + 4 < dim ? *reinterpret_cast<const float4*>(from + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
            const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
            half8v h;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                h[e] = static_cast<_Float16>(v[e] * scale);
                const float d = fmaf(-unit, static_cast<float>(h[e]), v[e]);
                off = fmaf(d, d, off);
                length = fmaf(v[e], v[e], length);
            }
            *reinterpret_cast<half8v*>(out + row * stride + d0) = h;
        }
#pragma unroll
        for (int w = 8; w > 0; w >>= 1) {
            off += __shfl_xor(off, w);
            length += __shfl_xor(length, w);
        }
        float r = kRoughTurn;   // lengths whose squares leave the range say nothing
        if (length > 1e-24f && length < 1e37f) r = fminf(fmaxf(sqrtf(off) * 1.001f - t, 0.f) / sqrtf(length) * 1.001f, kRoughTurn);
        most = fmaxf(most, r);
    }
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) most = fmaxf(most, __shfl_xor(most, w));
    __shared__ float of_wave[4];
    if (lane_id() == 0) of_wave[threadIdx.x >> 6] = most;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(turn_bits, __float_as_uint(fmaxf(fmaxf(of_wave[0], of_wave[1]), fmaxf(of_wave[2], of_wave[3]))));
}

// Whether a first look in fp16 will settle anything, from some rows and the graph that their searches will go through; four
// wavefronts a row, which have all rows of a list under way at once.  counts[0] / counts[1]: neighbours of a neighbour that are
// farther than the row's own farthest one, and how many of them the look's bounds would tell to be so.  counts[2] / counts[3]: rows,
// and those that a greedy walk from their segment's start ends one and a half times that far from, or more: searches that do not get to
// where they should stay among few rows, the caches serve those, and the look has no traffic to save.  A chain of two round trips a
// list: with the counts read back 50 to 60 us on rows of 128 to 512 values, 72 on 960 (one wavefront a row, 512 rows and all of up to 64
// neighbours: 70 to 110, and 190 at degree 64; 1.3 % of a build of 13 000 x 512).
struct SurveyArgs {
    const float* rows;
    const unsigned char* rough;
    const uint32_t *graph, *starts, *lengths, *start_points;
    uint32_t num, dim, degree, segment_num;
    uint32_t* counts;
};
constexpr uint32_t kSurveyed = 256, kSurveyWaves = 4, kSurveyDegree = 32, kMostHops = 64;
template <int DIMV>
__global__ __launch_bounds__(64 * kSurveyWaves) void rough_survey_kernel(SurveyArgs a) {
    __shared__ uint32_t own[kSurveyDegree], list[kSurveyDegree];
    __shared__ float sq[kSurveyDegree];
    const int lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t row = static_cast<uint32_t>(static_cast<unsigned long long>(blockIdx.x) * a.num / gridDim.x);
    uint32_t seg = kInvalid;
    for (uint32_t s0 = 0; s0 < a.segment_num && seg == kInvalid; s0 += 64) {
        const uint32_t s = s0 + lane;
        const uint64_t m = ballot(s < a.segment_num && row - a.starts[s] < a.lengths[s]);   // below the start it wraps
        if (m != 0) seg = s0 + __builtin_ctzll(m);
    }
    if (seg == kInvalid) return;
    const uint32_t first = a.starts[seg], length = a.lengths[seg], self = row - first, degree = a.degree < kSurveyDegree ? a.degree : kSurveyDegree;
    const float* data = a.rows + static_cast<size_t>(first) * a.dim;
    RowRegs<DIMV> q;
    load_row<DIMV>(q, a.rows + static_cast<size_t>(row) * a.dim, a.dim, RowShape<DIMV>::lane_in_row(lane));
    // this lane's neighbour of a row of the segment, kInvalid if none or the row itself, and its squared distance
    auto look_at = [&](uint32_t of, float& d) {
        uint32_t id = static_cast<uint32_t>(lane) < degree ? a.graph[static_cast<size_t>(first + of) * a.degree + lane] : kInvalid;
        if (id >= length || id == self) id = kInvalid;
        if (wave == 0 && static_cast<uint32_t>(lane) < degree) list[lane] = id != kInvalid ? id : self;
        __syncthreads();
        score_share<DIMV, DIMV < 4 ? DIMV : 4>(RefInRegs<DIMV>{q}, data, a.dim, 0, degree, lane, wave, kSurveyWaves, [](uint32_t i) { return list[i]; },
                             [](uint32_t i, float v) { sq[i] = v; });
        __syncthreads();   // the next list is written behind the reads below: by wavefront 0, which has made them; sq behind a barrier more
        d = id != kInvalid ? sq[lane] : __builtin_inff();
        return id;
    };
    float d;
    const uint32_t id = look_at(self, d);
    if (wave == 0 && static_cast<uint32_t>(lane) < degree) own[lane] = id;   // read behind the barriers of the next list
    uint64_t some = ballot(id != kInvalid);
    if (some == 0) return;
    float farthest = id != kInvalid ? d : 0.f;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) farthest = fmaxf(farthest, __shfl_xor(farthest, m));
    for (int drop = __popcll(some) / 2; drop > 0; drop--) some &= some - 1;
    const uint32_t of_middle = look_at(read_lane(id, __builtin_ctzll(some)), d);
    bool far = of_middle != kInvalid && d >= farthest;
    for (uint32_t j = 0; j < degree; j++) far &= own[j] != of_middle;
    const RoughRows look = rough_rows(a.rough, a.dim);
    const float off = 2 * look.turn * row_length<DIMV>(q) + look.tiny;   // a sum over lanes: every lane takes part
    const bool settled = far && sqrtf(d) * (1.f - 2 * kRoughTurn) - off >= sqrtf(farthest);
    const uint32_t fars = __popcll(ballot(far)), settleds = __popcll(ballot(settled));
    float nearest = __builtin_inff();
    uint32_t at = a.start_points[seg] < length ? a.start_points[seg] : 0u;
    for (uint32_t hop = 0; hop < kMostHops; hop++) {
        const uint32_t next = look_at(at, d);
        float least = d;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) least = fminf(least, __shfl_xor(least, m));
        if (!(least < nearest)) break;
        nearest = least;
        at = read_lane(next, __builtin_ctzll(ballot(d == least)));
    }
    if (threadIdx.x == 0) {
        atomicAdd(&a.counts[0], fars);
        atomicAdd(&a.counts[1], settleds);
        atomicAdd(&a.counts[2], 1u);
        if (!(nearest <= 2.25f * farthest)) atomicAdd(&a.counts[3], 1u);
    }
}

// ------------------------------------------------------------------------------------------ merged large build
// A staged partition's sub-graph holds partition-local ids.  Its rows go to rows segment_start .. of the merged graph
// with segment_start added to every id (what map_to_graph does through `map` on the small path,
// graph_kernel.cuh:145-150; here the merged graph stays in reorder-id space, so the map is an offset).
__global__ __launch_bounds__(256) void place_segment_kernel(const uint32_t* segment_graph, size_t words, uint32_t segment_start, uint32_t* merged) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= words) return;
    const uint32_t v = segment_graph[i];
    merged[i] = v == kInvalid ? kInvalid : v + segment_start;
}

// map_to_graph_boundary (graph_kernel.cuh:160-247) as a pass of its own: boundary copy i found the neighbours
// boundary_graph[i] (ids local to the boundary segment); they are merged into the row of the point it is a copy of,
// home_rows[i], every neighbour l being named by its own home row home_rows[l].  One wavefront per boundary copy.
__global__ __launch_bounds__(64) void merge_boundary_kernel(const uint32_t* boundary_graph, uint32_t boundary_num, uint32_t D,
                                                            const uint32_t* home_rows, uint32_t* merged) {
    __shared__ PruneLds<64> pl;
    const uint32_t i = blockIdx.x;
    if (i >= boundary_num) return;
    const int lane = lane_id();
    for (uint32_t j = lane; j < kMaxDegree; j += 64) pl.neighbor[j] = j < D ? boundary_graph[static_cast<size_t>(i) * D + j] : kInvalid;
    wave_sync();
    merge_boundary_row<64>(&pl, merged + static_cast<size_t>(home_rows[i]) * D, home_rows, D, lane);
}

// ------------------------------------------------------------------------------------------ dispatch
size_t prune_lds_bytes(uint32_t beam) {
    return beam <= 64 ? sizeof(PruneLds<64>) : beam <= 128 ? sizeof(PruneLds<128>) : beam <= 256 ? sizeof(PruneLds<256>) : sizeof(PruneLds<512>);
}
// the refine kernel's layout: row arrays sized by the degree bucket instead of the maximum degree
template <int CAP>
size_t prune_lds_bytes_cap(uint32_t beam) {
    return beam <= 64 ? sizeof(PruneLds<64, CAP>) : beam <= 128 ? sizeof(PruneLds<128, CAP>) : beam <= 256 ? sizeof(PruneLds<256, CAP>)
                                                                                                          : sizeof(PruneLds<512, CAP>);
}
size_t prune_lds_bytes_refine(uint32_t beam, uint32_t degree) {
    return degree <= 64 ? prune_lds_bytes_cap<64>(beam) : degree <= 128 ? prune_lds_bytes_cap<128>(beam) : prune_lds_bytes_cap<256>(beam);
}

int check_beam_sizes(uint32_t degree, uint32_t graph_degree, uint32_t beam, uint32_t dim, uint32_t hash_bit, int metric) {
    if (degree == 0 || graph_degree == 0 || beam == 0 || dim == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (metric != GLIDE_METRIC_EUCLIDEAN && metric != GLIDE_METRIC_COSINE) return GLIDE_ERR_BAD_ARGUMENT;
    if (degree > kMaxDegree || graph_degree > kMaxDegree || !beam_supported(beam) || dim % 4 != 0 || dim > 4096 || hash_bit < 1 || hash_bit > 13)
        return GLIDE_ERR_UNSUPPORTED;
    return GLIDE_OK;
}

bool byte_rows_serve(const unsigned char* bytes, uint32_t degree, uint32_t dim) { return bytes && degree <= kMostByteDegree && dim <= kMostByteDims; }

// the bounds of the prune want a factor that keeps their order
bool rough_rows_serve(const unsigned char* rough, uint32_t degree, uint32_t beam, uint32_t dim, float relaxant) {
    return rough && degree <= 64 && beam <= kMostRoughBeam && dim <= kMostRoughDims && relaxant > 0.f && relaxant < 1e18f;
}

int launch_build(BuildArgs& a, hipStream_t stream) {
    if (reinterpret_cast<uintptr_t>(a.bytes) % 16 || reinterpret_cast<uintptr_t>(a.rough) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    build_fn fn = byte_rows_serve(a.bytes, a.p.degree, a.p.dim)                              ? pick_build_bytes(a.p.beam, a.p.dim)
                  : rough_rows_serve(a.rough, a.p.degree, a.p.beam, a.p.dim, a.relaxant) ? pick_build_rough(a.p.beam, a.p.dim)
                                                                                             : pick_build(a.p.degree, a.p.beam, a.p.dim);
    const size_t lds_bytes = beam_lds_bytes(a.p.degree) + prune_lds_bytes(a.p.beam) + (size_t{1} << a.p.hash_bit) * sizeof(uint32_t);
    GLIDE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
    hipLaunchKernelGGL(fn, dim3(a.point_count), dim3(64), lds_bytes, stream, a);
    return launch_status();
}

}  // namespace glide

using namespace glide;

extern "C" {

int glide_hip_build_subgraph(const float* reorder_data, uint32_t num, uint32_t dim, const uint32_t* knn_graph, uint32_t knn_degree,
                             const uint32_t* map, const uint32_t* segment_starts, const uint32_t* segment_lengths,
                             uint32_t segment_num, const uint32_t* start_points, uint32_t graph_degree, uint32_t beam,
                             uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit, uint32_t hash_reset_interval,
                             float relaxant, int metric, uint32_t* graph, unsigned long long* counters, void* stream) {
    return glide_hip_build_subgraph_rows(reorder_data, nullptr, nullptr, num, dim, knn_graph, knn_degree, map, segment_starts, segment_lengths, segment_num,
                                         start_points, graph_degree, beam, max_iterations, min_iterations, hash_bit, hash_reset_interval, relaxant,
                                         metric, graph, counters, stream);
}

int glide_hip_build_subgraph_rows(const float* reorder_data, const void* byte_rows, const void* rough_rows, uint32_t num, uint32_t dim,
                                  const uint32_t* knn_graph, uint32_t knn_degree, const uint32_t* map, const uint32_t* segment_starts, const uint32_t* segment_lengths,
                                  uint32_t segment_num, const uint32_t* start_points, uint32_t graph_degree, uint32_t beam,
                                  uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit, uint32_t hash_reset_interval,
                                  float relaxant, int metric, uint32_t* graph, unsigned long long* counters, void* stream) {
    if (!reorder_data || !knn_graph || !map || !segment_starts || !segment_lengths || !start_points || !graph)
        return GLIDE_ERR_BAD_ARGUMENT;
    if (max_iterations == 0 || segment_num == 0) return GLIDE_ERR_BAD_ARGUMENT;
    int rc = check_beam_sizes(knn_degree, graph_degree, beam, dim, hash_bit, metric);
    if (rc != GLIDE_OK) return rc;
    if (num == 0) return GLIDE_OK;
    BuildArgs a;
    a.reorder_data = reorder_data;
    a.bytes = static_cast<const unsigned char*>(byte_rows);
    a.rough = static_cast<const unsigned char*>(rough_rows);
    a.knn_graph = knn_graph;
    a.map = map;
    a.segment_starts = segment_starts;
    a.segment_lengths = segment_lengths;
    a.start_points = start_points;
    a.graph = graph;
    a.counters = counters;
    a.first_point = 0;
    a.point_count = num;
    a.segment_num = segment_num;
    a.graph_degree = graph_degree;
    a.boundary_start = kInvalid;
    a.boundary_start_point = 0;
    a.relaxant = relaxant;
    a.p = BeamParams{beam, knn_degree, dim, hash_bit, hash_reset_interval ? hash_reset_interval : 1, max_iterations, min_iterations, metric};
    return launch_build(a, as_stream(stream));
}

int glide_hip_build_boundary(const float* reorder_data, uint32_t num, uint32_t reorder_num, uint32_t dim, const uint32_t* knn_graph,
                             uint32_t knn_degree, const uint32_t* map, uint32_t start_point, uint32_t graph_degree, uint32_t beam,
                             uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit, uint32_t hash_reset_interval,
                             float relaxant, int metric, uint32_t* graph, unsigned long long* counters, void* stream) {
    return glide_hip_build_boundary_rows(reorder_data, nullptr, nullptr, num, reorder_num, dim, knn_graph, knn_degree, map, start_point, graph_degree, beam,
                                          max_iterations, min_iterations, hash_bit, hash_reset_interval, relaxant, metric, graph, counters, stream);
}

int glide_hip_build_boundary_rows(const float* reorder_data, const void* byte_rows, const void* rough_rows, uint32_t num, uint32_t reorder_num, uint32_t dim,
                                  const uint32_t* knn_graph, uint32_t knn_degree, const uint32_t* map, uint32_t start_point,
                                  uint32_t graph_degree, uint32_t beam, uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                                  uint32_t hash_reset_interval, float relaxant, int metric, uint32_t* graph, unsigned long long* counters,
                                  void* stream) {
    if (!reorder_data || !knn_graph || !map || !graph) return GLIDE_ERR_BAD_ARGUMENT;
    if (max_iterations == 0 || reorder_num < num) return GLIDE_ERR_BAD_ARGUMENT;
    int rc = check_beam_sizes(knn_degree, graph_degree, beam, dim, hash_bit, metric);
    if (rc != GLIDE_OK) return rc;
    if (reorder_num == num) return GLIDE_OK;
    if (start_point >= reorder_num - num) return GLIDE_ERR_BAD_ARGUMENT;
    BuildArgs a;
    a.reorder_data = reorder_data;
    a.bytes = static_cast<const unsigned char*>(byte_rows);
    a.rough = static_cast<const unsigned char*>(rough_rows);
    a.knn_graph = knn_graph;
    a.map = map;
    a.segment_starts = nullptr;
    a.segment_lengths = nullptr;
    a.start_points = nullptr;
    a.graph = graph;
    a.counters = counters;
    a.first_point = num;
    a.point_count = reorder_num - num;
    a.segment_num = 0;
    a.graph_degree = graph_degree;
    a.boundary_start = num;
    a.boundary_start_point = start_point;
    a.relaxant = relaxant;
    a.p = BeamParams{beam, knn_degree, dim, hash_bit, hash_reset_interval ? hash_reset_interval : 1, max_iterations, min_iterations, metric};
    return launch_build(a, as_stream(stream));
}

int glide_hip_build_segment(const float* segment_data, uint32_t num, uint32_t dim, const uint32_t* knn_graph, uint32_t knn_degree,
                            uint32_t start_point, uint32_t graph_degree, uint32_t beam, uint32_t max_iterations, uint32_t min_iterations,
                            uint32_t hash_bit, uint32_t hash_reset_interval, float relaxant, int metric, uint32_t* graph,
                            unsigned long long* counters, void* stream) {
    if (!segment_data || !knn_graph || !graph) return GLIDE_ERR_BAD_ARGUMENT;
    if (max_iterations == 0) return GLIDE_ERR_BAD_ARGUMENT;
    int rc = check_beam_sizes(knn_degree, graph_degree, beam, dim, hash_bit, metric);
    if (rc != GLIDE_OK) return rc;
    if (num == 0) return GLIDE_OK;
    if (start_point >= num) return GLIDE_ERR_BAD_ARGUMENT;
    BuildArgs a;
    a.reorder_data = segment_data;
    a.bytes = nullptr;
    a.rough = nullptr;
    a.knn_graph = knn_graph;
    a.map = nullptr;
    a.segment_starts = nullptr;
    a.segment_lengths = nullptr;
    a.start_points = nullptr;
    a.graph = graph;
    a.counters = counters;
    a.first_point = 0;
    a.point_count = num;
    a.segment_num = 0;
    a.graph_degree = graph_degree;
    a.boundary_start = kInvalid;
    a.boundary_start_point = start_point;
    a.relaxant = relaxant;
    a.p = BeamParams{beam, knn_degree, dim, hash_bit, hash_reset_interval ? hash_reset_interval : 1, max_iterations, min_iterations, metric};
    return launch_build(a, as_stream(stream));
}

int glide_hip_refine_segment(const float* segment_data, uint32_t num, uint32_t dim, const uint32_t* graph_in, uint32_t* graph_out,
                             uint32_t graph_degree, uint32_t start_point, uint32_t beam, uint32_t max_iterations, uint32_t min_iterations,
                             uint32_t hash_bit, uint32_t hash_reset_interval, float relaxant, int metric, unsigned long long* counters,
                             void* stream) {
    if (!segment_data || !graph_in || !graph_out || graph_in == graph_out) return GLIDE_ERR_BAD_ARGUMENT;
    if (max_iterations == 0) return GLIDE_ERR_BAD_ARGUMENT;
    int rc = check_beam_sizes(graph_degree, graph_degree, beam, dim, hash_bit, metric);
    if (rc != GLIDE_OK) return rc;
    if (num == 0) return GLIDE_OK;
    if (start_point >= num) return GLIDE_ERR_BAD_ARGUMENT;
    RefineArgs a;
    a.order = nullptr;
    a.data = segment_data;
    a.bytes = nullptr;
    a.rough = nullptr;
    a.graph_in = graph_in;
    a.graph_out = graph_out;
    a.centroids = nullptr;
    a.start_points = nullptr;
    a.counters = counters;
    a.num = num;
    a.centroid_num = 0;
    a.max_centroid = 32;
    a.segment_start_point = start_point;
    a.relaxant = relaxant;
    a.p = BeamParams{beam, graph_degree, dim, hash_bit, hash_reset_interval ? hash_reset_interval : 1, max_iterations, min_iterations, metric};
    refine_fn fn = pick_refine(graph_degree, beam, dim);
    const size_t lds_bytes = beam_lds_bytes(graph_degree) + prune_lds_bytes(beam) + (size_t{1} << hash_bit) * sizeof(uint32_t);
    GLIDE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
    hipLaunchKernelGGL(fn, dim3(num), dim3(64), lds_bytes, as_stream(stream), a);
    return launch_status();
}

size_t glide_hip_reverse_edges_workspace_bytes(uint32_t num, uint32_t graph_degree) {
    const size_t n = num, words = ceil_div(graph_degree, 32);
    // miss bits + offsets + fill (u32 each), cursor (u64, 256-byte slot), pool of (column, source) keys
    return n * words * 4 + n * 4 + n * 4 + 256 + n * graph_degree * 8;
}

int glide_hip_reverse_edges(const uint32_t* graph, uint32_t num, uint32_t graph_degree, uint32_t* reverse_graph,
                            uint32_t* reverse_counts, void* workspace, size_t workspace_bytes, void* stream) {
    if (!graph || !reverse_graph || !reverse_counts || !workspace) return GLIDE_ERR_BAD_ARGUMENT;
    if (graph_degree == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (graph_degree > 256) return GLIDE_ERR_UNSUPPORTED;
    if (num == 0) return GLIDE_OK;
    if (workspace_bytes < glide_hip_reverse_edges_workspace_bytes(num, graph_degree) || reinterpret_cast<uintptr_t>(workspace) % 8)
        return GLIDE_ERR_BAD_ARGUMENT;
    hipStream_t s = as_stream(stream);
    const size_t n = num, words = ceil_div(graph_degree, 32);
    unsigned char* w = static_cast<unsigned char*>(workspace);
    unsigned long long* cursor = reinterpret_cast<unsigned long long*>(w);
    unsigned long long* pool = reinterpret_cast<unsigned long long*>(w + 256);
    uint32_t* offsets = reinterpret_cast<uint32_t*>(w + 256 + n * graph_degree * 8);
    uint32_t* fill = offsets + n;
    uint32_t* miss = fill + n;
    int rc = glide_hip_fill_u32(reverse_counts, 0u, n, stream);
    if (rc == GLIDE_OK) rc = glide_hip_fill_u32(fill, 0u, n, stream);
    if (rc == GLIDE_OK) rc = glide_hip_fill_u32(reinterpret_cast<uint32_t*>(cursor), 0u, 2, stream);
    if (rc != GLIDE_OK) return rc;
    hipLaunchKernelGGL(reverse_count_kernel, dim3(ceil_div(num, 4)), dim3(256), 0, s, graph, num, graph_degree, miss, reverse_counts);
    hipLaunchKernelGGL(reverse_offsets_kernel, dim3(ceil_div(num, 256)), dim3(256), 0, s, reverse_counts, num, offsets, cursor);
    hipLaunchKernelGGL(reverse_scatter_kernel, dim3(ceil_div(num, 256)), dim3(256), 0, s, graph, num, graph_degree, miss, offsets, fill, pool);
    hipLaunchKernelGGL(reverse_select_kernel, dim3(ceil_div(num, 4)), dim3(256), 0, s, num, graph_degree, reverse_counts, offsets, pool,
                       reverse_graph);
    (void) words;
    return launch_status();
}

int glide_hip_insert_reverse(uint32_t* graph, const uint32_t* reverse_graph, const uint32_t* reverse_counts, uint32_t num,
                             uint32_t graph_degree, void* stream) {
    if (!graph || !reverse_graph || !reverse_counts || graph_degree == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (num == 0) return GLIDE_OK;
    hipLaunchKernelGGL(insert_reverse_kernel, dim3(ceil_div(num, 4)), dim3(256), 0, as_stream(stream), graph, reverse_graph,
                       reverse_counts, num, graph_degree);
    return launch_status();
}

size_t glide_hip_byte_rows_bytes(uint32_t num, uint32_t dim) {
    if (dim == 0 || dim > kMostByteDims || dim % 4 != 0) return 0;
    const size_t bytes = static_cast<size_t>(num) * (dim <= 128 ? RowShape<-1>::STRIDE : RowShape<-2>::STRIDE);
    return bytes <= kMostPacked ? bytes : 0;
}

int glide_hip_pack_byte_rows(const float* rows, uint32_t num, uint32_t dim, void* byte_rows, uint32_t* other_values, void* stream) {
    if (!rows || !byte_rows || !other_values || dim == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (glide_hip_byte_rows_bytes(1, dim) == 0 || (num != 0 && glide_hip_byte_rows_bytes(num, dim) == 0)) return GLIDE_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(rows) % 16 || reinterpret_cast<uintptr_t>(byte_rows) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    const int rc = glide_hip_fill_u32(other_values, 0u, 1, stream);
    if (rc != GLIDE_OK || num == 0) return rc;
    const uint32_t lanes = dim <= 128 ? RowShape<-1>::LPR : RowShape<-2>::LPR;   // sixteen dims each
    const size_t blocks = (static_cast<size_t>(num) * lanes + 255) / 256;
    const uint32_t probe = blocks < kPackProbe ? static_cast<uint32_t>(blocks) : kPackProbe;
    hipLaunchKernelGGL(pack_bytes_kernel, dim3(probe), dim3(256), 0, as_stream(stream), rows, num, dim, lanes, 0u, static_cast<uint4*>(byte_rows),
                       other_values);
    if (blocks > probe)
        hipLaunchKernelGGL(pack_bytes_kernel, dim3(static_cast<uint32_t>(blocks) - probe), dim3(256), 0, as_stream(stream), rows, num, dim, lanes, probe,
                           static_cast<uint4*>(byte_rows), other_values);
    return launch_status();
}

size_t glide_hip_rough_rows_bytes(uint32_t num, uint32_t dim) {
    return dim > 0 && dim <= kMostRoughDims && dim % 4 == 0 ? kRoughHeader + static_cast<size_t>(num) * rough_stride(dim) * 2 : 0;
}

int glide_hip_pack_rough_rows(const float* rows, uint32_t num, uint32_t dim, void* rough_rows, void* stream) {
    if (!rows || !rough_rows || dim == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (glide_hip_rough_rows_bytes(1, dim) == 0) return GLIDE_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(rows) % 16 || reinterpret_cast<uintptr_t>(rough_rows) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    uint32_t* max_bits = static_cast<uint32_t*>(rough_rows);
    const int rc = glide_hip_fill_u32(max_bits, 0u, kRoughHeader / 4, stream);
    if (rc != GLIDE_OK || num == 0) return rc;
    const size_t quads = static_cast<size_t>(num) * (dim / 4);
    const uint32_t blocks = static_cast<uint32_t>(quads / 256 < 1024 ? quads / 256 + 1 : 1024), row_blocks = num < 16 * 2048 ? ceil_div(num, 16u) : 2048u;
    hipLaunchKernelGGL(rough_range_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), rows, quads, max_bits);
    hipLaunchKernelGGL(rough_pack_kernel, dim3(row_blocks), dim3(256), 0, as_stream(stream), rows, num, dim, max_bits, max_bits + 1,
                       reinterpret_cast<_Float16*>(static_cast<unsigned char*>(rough_rows) + kRoughHeader));
    return launch_status();
}

int glide_hip_survey_rough_rows(const float* rows, const void* rough_rows, uint32_t num, uint32_t dim, const uint32_t* graph, uint32_t degree,
                                const uint32_t* segment_starts, const uint32_t* segment_lengths, uint32_t segment_num, const uint32_t* start_points,
                                uint32_t* counts, void* stream) {
    if (!rows || !rough_rows || !graph || !segment_starts || !segment_lengths || !start_points || !counts || dim == 0 || degree == 0)
        return GLIDE_ERR_BAD_ARGUMENT;
    if (glide_hip_rough_rows_bytes(1, dim) == 0) return GLIDE_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(rows) % 16 || reinterpret_cast<uintptr_t>(rough_rows) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    const int rc = glide_hip_fill_u32(counts, 0u, 4, stream);
    if (rc != GLIDE_OK || num == 0) return rc;
    const SurveyArgs a{rows, static_cast<const unsigned char*>(rough_rows), graph, segment_starts, segment_lengths, start_points, num, dim, degree,
                       segment_num, counts};
    const auto kernel = dim <= 128 ? rough_survey_kernel<1> : dim <= 256 ? rough_survey_kernel<2> : dim <= 512 ? rough_survey_kernel<4> : rough_survey_kernel<8>;
    hipLaunchKernelGGL(kernel, dim3(num < kSurveyed ? num : kSurveyed), dim3(64 * kSurveyWaves), 0, as_stream(stream), a);
    return launch_status();
}

int glide_hip_place_segment_graph(const uint32_t* segment_graph, uint32_t segment_length, uint32_t graph_degree, uint32_t segment_start,
                                  uint32_t* merged_graph, void* stream) {
    if (!segment_graph || !merged_graph || graph_degree == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (segment_length == 0) return GLIDE_OK;
    const size_t words = static_cast<size_t>(segment_length) * graph_degree;
    uint32_t* dst = merged_graph + static_cast<size_t>(segment_start) * graph_degree;
    hipLaunchKernelGGL(place_segment_kernel, dim3(static_cast<uint32_t>((words + 255) / 256)), dim3(256), 0, as_stream(stream), segment_graph, words,
                       segment_start, dst);
    return launch_status();
}

int glide_hip_merge_boundary_graph(const uint32_t* boundary_graph, uint32_t boundary_num, uint32_t graph_degree, const uint32_t* home_rows,
                                   uint32_t* merged_graph, void* stream) {
    if (!boundary_graph || !home_rows || !merged_graph || graph_degree == 0) return GLIDE_ERR_BAD_ARGUMENT;
    if (graph_degree > kMaxDegree) return GLIDE_ERR_UNSUPPORTED;
    if (boundary_num == 0) return GLIDE_OK;
    hipLaunchKernelGGL(merge_boundary_kernel, dim3(boundary_num), dim3(64), 0, as_stream(stream), boundary_graph, boundary_num, graph_degree,
                       home_rows, merged_graph);
    return launch_status();
}

}  // extern "C"

namespace {
int launch_refine(const float* data, const unsigned char* bytes, const unsigned char* rough, uint32_t num, uint32_t dim, const uint32_t* graph_in, uint32_t* graph_out, uint32_t graph_degree,
                  const float* centroids, uint32_t centroid_num, bool rank_all_centroids, const uint32_t* start_points, uint32_t beam,
                  uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit, uint32_t hash_reset_interval, float relaxant, int metric,
                  const uint32_t* order, unsigned long long* counters, void* stream) {
    if (!data || !graph_in || !graph_out || !centroids || !start_points || graph_in == graph_out) return GLIDE_ERR_BAD_ARGUMENT;
    if (max_iterations == 0 || centroid_num == 0) return GLIDE_ERR_BAD_ARGUMENT;
    int rc = check_beam_sizes(graph_degree, graph_degree, beam, dim, hash_bit, metric);
    if (rc != GLIDE_OK) return rc;
    if (centroid_num > 256) return GLIDE_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(bytes) % 16 || reinterpret_cast<uintptr_t>(rough) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    if (num == 0) return GLIDE_OK;
    RefineArgs a;
    a.data = data;
    a.bytes = bytes;
    a.rough = rough;
    a.graph_in = graph_in;
    a.graph_out = graph_out;
    a.centroids = centroids;
    a.start_points = start_points;
    a.counters = counters;
    a.order = order;
    a.num = num;
    a.centroid_num = centroid_num;
    a.max_centroid = centroid_num <= 32 ? 32 : (graph_degree <= 64 ? 64 : (graph_degree <= 128 ? 128 : 256));
    if (rank_all_centroids) a.max_centroid = centroid_num <= 32 ? 32 : (centroid_num <= 64 ? 64 : (centroid_num <= 128 ? 128 : 256));
    a.segment_start_point = 0;
    a.relaxant = relaxant;
    a.p = BeamParams{beam, graph_degree, dim, hash_bit, hash_reset_interval ? hash_reset_interval : 1, max_iterations, min_iterations, metric};
    refine_fn fn = byte_rows_serve(bytes, graph_degree, dim)                           ? pick_refine_bytes(beam, dim)
                   : rough_rows_serve(rough, graph_degree, beam, dim, relaxant) ? pick_refine_rough(beam, dim)
                                                                                 : pick_refine(graph_degree, beam, dim);
    const size_t lds_bytes = beam_lds_bytes(graph_degree) + prune_lds_bytes_refine(beam, graph_degree) + round_up32(centroid_num) * sizeof(float) +
                             (size_t{1} << hash_bit) * sizeof(uint32_t);
    GLIDE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
    hipLaunchKernelGGL(fn, dim3(num), dim3(64), lds_bytes, as_stream(stream), a);
    return launch_status();
}
}  // namespace

extern "C" int glide_hip_refine(const float* data, uint32_t num, uint32_t dim, const uint32_t* graph_in, uint32_t* graph_out,
                                uint32_t graph_degree, const float* centroids, uint32_t centroid_num, const uint32_t* start_points,
                                uint32_t beam, uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                                uint32_t hash_reset_interval, float relaxant, int metric, const uint32_t* order,
                                unsigned long long* counters, void* stream) {
    return launch_refine(data, nullptr, nullptr, num, dim, graph_in, graph_out, graph_degree, centroids, centroid_num, false, start_points, beam, max_iterations,
                         min_iterations, hash_bit, hash_reset_interval, relaxant, metric, order, counters, stream);
}

extern "C" int glide_hip_refine_rows(const float* data, const void* byte_rows, const void* rough_rows, uint32_t num, uint32_t dim,
                                     const uint32_t* graph_in, uint32_t* graph_out, uint32_t graph_degree, const float* centroids, uint32_t centroid_num,
                                      const uint32_t* start_points, uint32_t beam, uint32_t max_iterations, uint32_t min_iterations,
                                      uint32_t hash_bit, uint32_t hash_reset_interval, float relaxant, int metric, const uint32_t* order,
                                      unsigned long long* counters, void* stream) {
    return launch_refine(data, static_cast<const unsigned char*>(byte_rows), static_cast<const unsigned char*>(rough_rows), num, dim, graph_in, graph_out, graph_degree, centroids, centroid_num, false,
                         start_points, beam, max_iterations, min_iterations, hash_bit, hash_reset_interval, relaxant, metric, order, counters, stream);
}

extern "C" int glide_hip_refine_merged(const float* data, uint32_t num, uint32_t dim, const uint32_t* graph_in, uint32_t* graph_out,
                                       uint32_t graph_degree, const float* centroids, uint32_t centroid_num, const uint32_t* start_points,
                                       uint32_t beam, uint32_t max_iterations, uint32_t min_iterations, uint32_t hash_bit,
                                       uint32_t hash_reset_interval, float relaxant, int metric, const uint32_t* order,
                                       unsigned long long* counters, void* stream) {
    return launch_refine(data, nullptr, nullptr, num, dim, graph_in, graph_out, graph_degree, centroids, centroid_num, true, start_points, beam, max_iterations,
                         min_iterations, hash_bit, hash_reset_interval, relaxant, metric, order, counters, stream);
}
