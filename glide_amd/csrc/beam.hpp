// Beam-search core for one item per 64-lane wavefront (search, sub-graph build, refine all use it).
//
// Reference semantics: search_kernel.cuh:433-482 / graph_kernel.cuh:16-63 (one iteration), :9-37 and :97-148
// (candidate sort, beam merge), :292-325 (parent selection), :327-334 (hash restore), :336-391 (expansion).
//
// Layout: the beam (MAX_BEAM entries) lives in registers, element e = NB*lane + r, ascending, explored flag in
// the id's MSB.  The D candidates of one expansion are produced into LDS by graph-row slot, pulled into
// registers with the reference's strided->blocked permutation, sorted by the wave network and staged back to
// LDS so that beam element e can pick candidate MAX_BEAM-1-e (the half-cleaner).  The visited set is an LDS
// open-addressing table.  Data rows are gathered several at a time (one lane group each, 16 B per lane and load).
#pragma once
#include "bitonic.hpp"

namespace glide {

struct BeamParams {
    uint32_t beam, degree, dim, hash_bit, reset_interval, max_iterations, min_iterations;
    int metric;
};

constexpr uint32_t kCounterStripes = 256;

// First result id of a query that a search over rows of bytes leaves to the fp32 kernel (result ids are below 2^31, or all ones).
constexpr uint32_t kLeftOver = 0xfffffffeu;

struct BeamCounters {  // wave-uniform tallies for traffic accounting
    uint32_t iterations = 0, rows_scored = 0, graph_rows = 0;
};

template <int MAX_CAND>
struct alignas(16) BeamLds {  // per-wave LDS (the hash table follows, 1 << hash_bit words)
    union {
        struct {
            uint32_t cand_id[MAX_CAND];
            float cand_dist[MAX_CAND];   // squared distances of vlist's rows while an expansion is scored, then distances by slot or rank
        };
        uint32_t pool_open[2 * MAX_CAND];   // once the search is over: see RoughPool
    };
    uint32_t vlist[MAX_CAND];    // row ids to score, compacted
};

// Beams the kernels take: up to 512 (the reference's widest bucket, kernel_config.cuh:41-48); above 256 a multiple of 16, so
// that each half of the beam is whole lanes of eight entries (the reference's adjust_search_params, params.cuh:82-99, only
// ever hands out multiples of 32).
inline bool beam_supported(uint32_t beam) { return beam <= 512 && (beam <= 256 || beam % 16 == 0); }

// Host-side size of the candidate lists for a degree bucket (the hash table follows them in the dynamic LDS).
inline size_t beam_lds_bytes(uint32_t degree) {
    return degree <= 64 ? sizeof(BeamLds<64>) : degree <= 128 ? sizeof(BeamLds<128>) : sizeof(BeamLds<256>);
}

__device__ __forceinline__ void wave_sync() { __syncthreads(); }  // workgroup == one wavefront
// The same point in a wavefront that shares its workgroup with others (TEAM): a workgroup barrier would wait for them.
// LDS instructions of one wavefront execute in program order; what is needed between a store and a dependent load of
// another lane is that the compiler keeps that order, which a wavefront-scope fence does.
template <bool TEAM>
__device__ __forceinline__ void wave_sync_in() {
    if constexpr (TEAM) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

// Where score_list reads the reference row from: registers (one copy per wavefront) ...
template <int DIMV>
struct RefInRegs {
    const RowRegs<DIMV>& r;
    __device__ __forceinline__ float sqdist(const RowRegs<DIMV>& row, int) const {
        if constexpr (RowShape<DIMV>::BYTES) return byte_sqdist<DIMV>(r, row.v);
        else return row_sum<DIMV>(partial_sqdist<DIMV>(r, row));
    }
};
// ... or LDS, laid out as the loads of one lane group would hold it (chunk c of lane t at [c * LPR + t]): the wavefronts
// of a team share one copy and keep their registers for rows in flight.  The two lane groups of a wide row read the same
// addresses (a broadcast), adjacent lanes adjacent 16-byte words: no bank conflicts.
template <int DIMV>
struct RefInLds {
    const float4* q;
    __device__ __forceinline__ float sqdist(const RowRegs<DIMV>& row, int t) const {
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < RowShape<DIMV>::NV; c++) acc = sqdist4(q[c * RowShape<DIMV>::LPR + t], row.v[c], acc);
        return row_sum<DIMV>(acc);
    }
};

// U steps of RowShape<DIMV>::ROWS rows each (one row per lane group): entries base .. base + ROWS * U of the list.
// FULL: the rows fill the row shape exactly, so no load needs a mask.
template <int DIMV, int U, bool FULL, class Ref, class IdFn, class OutFn>
__device__ __forceinline__ void score_step(const Ref ref, row_data<DIMV> data, uint32_t dim, uint32_t base, uint32_t count, int g, int t,
                                           IdFn id_of, OutFn out) {
    using Shape = RowShape<DIMV>;
    RowRegs<DIMV> rows[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        // lane groups past the end re-read the last listed row (same cache lines, no branch); their result is dropped
        const uint32_t idx = base + Shape::ROWS * u + g;
        load_row<DIMV, FULL>(rows[u], row_at<DIMV>(data, id_of(idx < count ? idx : count - 1), dim), dim, t);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t idx = base + Shape::ROWS * u + g;
        const float sq = ref.sqdist(rows[u], t);
        if (t == 0 && idx < count) out(idx, sq);
    }
}

// Squared distances from a reference row to `count` listed rows, U steps in flight.  id_of(idx) -> row id of list entry
// idx; out(idx, squared distance) is called by one lane per scored row (the root, some fifteen instructions, is left to
// the pass that reads the results with one lane per row).  A team of `members` wavefronts splits the list in runs of
// ROWS * U entries, member `member` taking every members-th run; the sum of a row is formed in the same order whoever
// forms it.  A run with at most half its entries takes half the steps: an expansion scores a dozen rows on average, and
// every step issues its loads and arithmetic whether its lane groups have rows or not.
template <int DIMV, int U, bool FULL, class Ref, class IdFn, class OutFn>
__device__ __forceinline__ void score_runs(const Ref ref, row_data<DIMV> data, uint32_t dim, uint32_t first, uint32_t count,
                                           int lane, uint32_t member, uint32_t members, IdFn id_of, OutFn out) {
    using Shape = RowShape<DIMV>;
    const int g = Shape::row_of_lane(lane), t = Shape::lane_in_row(lane);
    for (uint32_t base = first + member * Shape::ROWS * U; base < count; base += Shape::ROWS * U * members) {
        if constexpr (U > 2 && Shape::BYTES) {
            if (count - base <= Shape::ROWS) {
                score_step<DIMV, 1, FULL>(ref, data, dim, base, count, g, t, id_of, out);
                continue;
            }
        }
        if constexpr (U > 1) {
            if (count - base <= Shape::ROWS * (U / 2)) {
                score_step<DIMV, U / 2, FULL>(ref, data, dim, base, count, g, t, id_of, out);
                continue;
            }
        }
        score_step<DIMV, U, FULL>(ref, data, dim, base, count, g, t, id_of, out);
    }
}
template <int DIMV, int U, class Ref, class IdFn, class OutFn>
__device__ __forceinline__ void score_share(const Ref ref, row_data<DIMV> data, uint32_t dim, uint32_t first, uint32_t count,
                                            int lane, uint32_t member, uint32_t members, IdFn id_of, OutFn out) {
    // Rows of exactly 128 or 256 dims are the usual ones and their searches the ones the vector ALU bounds: no masks there.
    // Longer rows are bound by their bytes, a second copy of the loop would buy them nothing.
    if constexpr (DIMV == 1 || DIMV == 2) {
        if (dim == RowShape<DIMV>::LPR * RowShape<DIMV>::NV * 4) {
            score_runs<DIMV, U, true>(ref, data, dim, first, count, lane, member, members, id_of, out);
            return;
        }
    }
    score_runs<DIMV, U, false>(ref, data, dim, first, count, lane, member, members, id_of, out);
}

template <int DIMV, class IdFn, class OutFn>
__device__ __forceinline__ void score_list(const RowRegs<DIMV>& ref, row_data<DIMV> data, uint32_t dim,
                                           uint32_t first, uint32_t count, int lane, IdFn id_of, OutFn out) {
    // Steps in flight.  Rows of more than 512 dims are 2-4 KB each and a step holds only two of them: with one step in
    // flight a wavefront had 8 KB on its way, too little to cover the memory latency when a launch has about one
    // wavefront per SIMD (1 000 queries); four steps took the 960-dim beam-512 search from 16.8 to 13.2 ms.
    // A step of byte rows is one load: four of them (32 or 16 rows) on their way at once.
    constexpr int U = DIMV == 8 || RowShape<DIMV>::BYTES ? 4 : 2;   // rows of more than 1024 dims (DIMV 16, 32) take 64 registers a lane each: two steps
    score_share<DIMV, U>(RefInRegs<DIMV>{ref}, data, dim, first, count, lane, 0u, 1u, id_of, out);
}

// The same over the fp16 copy of the rows: out(idx, squared distance of the rounded rows).
template <int DIMV, int U, bool FULL, class IdFn, class OutFn>
__device__ __forceinline__ void rough_step(const RoughRegs<DIMV>& ref, const RoughRows& rough, uint32_t dim, uint32_t base, uint32_t count, int g, int t,
                                           IdFn id_of, OutFn out) {
    using Shape = RowShape<DIMV>;
    RoughRegs<DIMV> rows[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t idx = base + Shape::ROWS * u + g;
        load_rough<DIMV, FULL>(rows[u], rough, id_of(idx < count ? idx : count - 1), dim, t);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t idx = base + Shape::ROWS * u + g;
        const float sq = row_sum<DIMV>(rough_sqdist(ref, rows[u])) * rough.unit * rough.unit;
        if (t == 0 && idx < count) out(idx, sq);
    }
}
template <int DIMV, bool FULL, class IdFn, class OutFn>
__device__ __forceinline__ void rough_runs(const RoughRegs<DIMV>& ref, const RoughRows& rough, uint32_t dim, uint32_t first, uint32_t count, int lane,
                                           IdFn id_of, OutFn out) {
    using Shape = RowShape<DIMV>;
    constexpr int U = DIMV == 8 ? 8 : 4;   // twice the rows of the exact pass under way
    const int g = Shape::row_of_lane(lane), t = Shape::lane_in_row(lane);
    for (uint32_t base = first; base < count; base += Shape::ROWS * U) {
        if (count - base <= Shape::ROWS * (U / 2)) rough_step<DIMV, U / 2, FULL>(ref, rough, dim, base, count, g, t, id_of, out);
        else rough_step<DIMV, U, FULL>(ref, rough, dim, base, count, g, t, id_of, out);
    }
}
template <int DIMV, class IdFn, class OutFn>
__device__ __forceinline__ void rough_list(const RoughRegs<DIMV>& ref, const RoughRows& rough, uint32_t dim, uint32_t first, uint32_t count, int lane,
                                           IdFn id_of, OutFn out) {
    if constexpr (DIMV == 1 || DIMV == 2) {   // as in score_share
        if (dim == RowShape<DIMV>::LPR * RowShape<DIMV>::NV * 4) {
            rough_runs<DIMV, true>(ref, rough, dim, first, count, lane, id_of, out);
            return;
        }
    }
    rough_runs<DIMV, false>(ref, rough, dim, first, count, lane, id_of, out);
}
// the reference row's length, or a little more, for the bounds of the rough distances
template <int DIMV>
__device__ __forceinline__ float row_length(const RowRegs<DIMV>& r) {
    float acc = 0.f;
#pragma unroll
    for (int c = 0; c < RowShape<DIMV>::NV; c++) acc = fmaf(r.v[c].x, r.v[c].x, fmaf(r.v[c].y, r.v[c].y, fmaf(r.v[c].z, r.v[c].z, fmaf(r.v[c].w, r.v[c].w, acc))));
    return sqrtf(row_sum<DIMV>(acc)) * 1.001f;
}

// TEAM: the beam's wavefront is one of several in its workgroup (the others only score rows, see search_team_kernel).
// WHOLE: the host promises beam == MAX_BEAM (asked for beams above 256 only, i.e. beam 512): the two-half merge of such a
// beam needs no lane permutations and tracks no turning points (merge_beam_full).
// ROUGH: rows are looked at in fp16 first (one candidate slot a lane).  Sub-graph builds and refinement over rows that are not in
// the caches run at the memory's rate: with nine tenths of the rows read in half the bytes, 120 000 rows of 512 values build in
// 87 ms instead of 136, 250 000 of 128 in 59 instead of 75, 60 000 of 960 (degree 64) in 225 instead of 355.
template <int MAX_CAND, int MAX_BEAM, int DIMV, bool TEAM = false, bool WHOLE = false, bool ROUGH = false>
struct Beam {
    static_assert(!ROUGH || (MAX_CAND == 64 && MAX_BEAM <= 128), "the lists of entries to measure are sized for these");
    static_assert(!WHOLE || MAX_BEAM > 256, "beams up to 256 merge in the registers anyway");
    static __device__ __forceinline__ void wave_sync() { wave_sync_in<TEAM>(); }
    static constexpr int NB = MAX_BEAM / 64;
    static constexpr int NC = MAX_CAND / 64;   // candidate slots per lane: slot 64 * i + lane
    static constexpr int NC32 = MAX_CAND / 32;  // items per lane in the reference's 32-lane layout

    float bk[NB];
    uint32_t bv[NB];
    RowRegs<DIMV> q;
    BeamLds<MAX_CAND>* lds;
    uint32_t* hash;
    BeamParams p;
    BeamCounters cnt;
    int lane;
    uint32_t last_scored;   // rows scored by the latest expansion (wave-uniform)
    uint32_t until_reset;   // iterations left until the visited set is reset (a countdown: a remainder by a run-time divisor is two dozen instructions)
    bool tied;              // some beam entries have equal keys (MAX_CAND == 64)
    // Entering candidates that are ranked rather than sorted (MAX_CAND == 64), or kUnordered: the beam holds rows that compare
    // with nothing, and no others (see absorb).  One number, so that the loop carries no second flag: that costs 1-2 %.
    static constexpr int kUnordered = -1;
    int rank_most;
    uint32_t cid;           // candidate id of this lane's slot (MAX_CAND == 64; larger buckets keep the ids in LDS)
    uint32_t place[NC];     // where in vlist each of this lane's slots is; kInvalid: not scored
    RoughRows rough;        // ROUGH: the rows in fp16,
    RoughRegs<ROUGH ? DIMV : 1> rough_q;
    float q_length;         // the reference row's length,
    uint64_t passed_over;   // and which entries of vlist a first look has found too far to enter (they count as infinitely far)

    __device__ __forceinline__ void begin(BeamLds<MAX_CAND>* lds_, uint32_t* hash_, const BeamParams& p_) {
        lds = lds_;
        hash = hash_;
        p = p_;
        lane = lane_id();
        asm volatile("" : "+v"(lane));   // as in run: nothing made from it is to be kept from one query to the next
        until_reset = p.reset_interval;
    }
    __device__ __forceinline__ void init(BeamLds<MAX_CAND>* lds_, uint32_t* hash_, const BeamParams& p_, row_data<DIMV> query) {
        begin(lds_, hash_, p_);
        load_reference<DIMV>(q, query, p.dim, RowShape<DIMV>::lane_in_row(lane));
        hash_clear(hash, p.hash_bit, lane);
        wave_sync();
    }
    // An fp32 query against rows of bytes; false if it is not of bytes itself.
    __device__ __forceinline__ bool init_packing(BeamLds<MAX_CAND>* lds_, uint32_t* hash_, const BeamParams& p_, const float* query) {
        static_assert(RowShape<DIMV>::BYTES, "rows of bytes");
        begin(lds_, hash_, p_);
        const bool exact = pack_bytes(query, 16 * RowShape<DIMV>::lane_in_row(lane), p.dim, q.v);
        if (ballot(!exact) != 0) return false;
        q.sq = dot_bytes(q.v, q.v, 0u);
        hash_clear(hash, p.hash_bit, lane);
        wave_sync();
        return true;
    }

    // whether this iteration ends with a reset of the visited set
    __device__ __forceinline__ bool count_down() {
        if (--until_reset != 0) return false;
        until_reset = p.reset_interval;
        return true;
    }

    // One pass of the main loop up to the next expansion's candidate list (what `run` does between two score phases).
    // Returns false when the search is over; otherwise `nv` rows wait to be scored.
    __device__ __forceinline__ bool step_to_list(uint32_t& iter, bool& terminate, const uint32_t* graph, uint32_t self_id, uint32_t& nv) {
        absorb(iter == 0, nullptr);
        cnt.iterations++;
        const bool reset_now = count_down();
        if (reset_now) {
            hash_clear(hash, p.hash_bit, lane);
            wave_sync();
        }
        if (iter + 1 == p.max_iterations) return false;
        const uint32_t parent = select_parent();
        if (parent == kInvalid) terminate = true;
        if (reset_now) {
            restore_hash();
            wave_sync();
        }
        if (terminate && iter >= p.min_iterations) return false;
        nv = expand_list(parent, graph, self_id, kInvalid);
        iter++;
        return true;
    }

    // Expansion of `parent` (reference compute_distance / get_init / result_init second half):
    // every neighbour not yet in the visited set becomes a candidate; `exclude_insert` is never inserted,
    // `exclude_score` is inserted and kept as a candidate id but gets distance FLT_MAX.
    // First half: the candidate slots and the list of rows to score (returns its length).  vlist holds the row ids
    // themselves, one LDS read before the row loads instead of two that depend on each other.
    __device__ __forceinline__ uint32_t expand_list(uint32_t parent, const uint32_t* graph, uint32_t exclude_insert, uint32_t exclude_score) {
        uint32_t nv = 0;
        if (parent != kInvalid) cnt.graph_rows++;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const uint32_t s = 64 * i + lane;
            uint32_t nid = kInvalid;
            if (s < p.degree && parent != kInvalid) nid = graph[static_cast<size_t>(parent) * p.degree + s];
            const uint32_t flag = (nid != kInvalid && nid != exclude_insert) ? hash_insert(hash, p.hash_bit, nid) : 0;
            const uint32_t c = flag ? nid : kInvalid;
            if constexpr (NC == 1) cid = c;
            else lds->cand_id[s] = c;
            const bool score = c != kInvalid && c != exclude_score;
            const uint64_t m = ballot(score);
            place[i] = score ? nv + prefix_count(m) : kInvalid;
            if (score) lds->vlist[place[i]] = c;
            nv += __popcll(m);
        }
        wave_sync();
        cnt.rows_scored += nv;
        last_scored = nv;
        return nv;
    }

    // exact squared distances of the entries of vlist named by a lane mask
    __device__ __forceinline__ void measure(uint64_t which, row_data<DIMV> data) {
        static_assert(!ROUGH || MAX_CAND == 64, "one entry a lane");
        if (which == 0) {
            wave_sync();
            return;
        }
        BeamLds<MAX_CAND>* l = lds;
        if ((which >> lane) & 1) l->cand_id[prefix_count(which)] = lane;   // the ids of a search with one slot a lane are in registers: the list is free
        wave_sync();
        score_list<DIMV>(q, data, p.dim, 0, __popcll(which), lane,
                         [l](uint32_t idx) { return l->vlist[l->cand_id[idx]]; },
                         [l](uint32_t idx, float sq) { l->cand_dist[l->cand_id[idx]] = sq; });
        wave_sync();
    }

    // `id`: the reference's row in `all`; the search's own ids start at `first`
    __device__ __forceinline__ void look_first(const RoughRows& all, uint32_t id, uint32_t first) {
        static_assert(ROUGH, "no fp16 rows");
        load_rough<DIMV, false>(rough_q, all, id, p.dim, RowShape<DIMV>::lane_in_row(lane));
        rough = all;
        rough.rows += static_cast<size_t>(first) * all.stride;
        q_length = row_length<DIMV>(q);
    }

    // `entry`: the first expansion of a search, whose beam holds nothing yet
    __device__ __forceinline__ void expand(uint32_t parent, const uint32_t* graph, row_data<DIMV> data,
                                           uint32_t exclude_insert, uint32_t exclude_score, bool entry = true) {
        const uint32_t nv = expand_list(parent, graph, exclude_insert, exclude_score);
        BeamLds<MAX_CAND>* l = lds;
        if constexpr (ROUGH) {
            passed_over = 0;
            const float tail = __uint_as_float(tail_key());
            if (!entry && nv != 0 && tail < FLT_MAX) {   // a beam that is not full takes every row
                rough_list<DIMV>(rough_q, rough, p.dim, 0, nv, lane,
                                 [l](uint32_t idx) { return l->vlist[idx]; },
                                 [l](uint32_t idx, float sq) { l->cand_dist[idx] = sq; });
                wave_sync();
                const float least = rough_least(rough, l->cand_dist[lane], q_length);
                const bool mine = static_cast<uint32_t>(lane) < nv;
                const bool out = mine && least > 0.f && (p.metric == kEuclidean ? least : least * least * (1.f - rough.slack)) >= tail;
                passed_over = ballot(out);
                if (out) l->cand_dist[lane] = __builtin_inff();
                measure(ballot(mine && !out), data);
                return;
            }
        }
        score_list<DIMV>(q, data, p.dim, 0, nv, lane,
                         [l](uint32_t idx) { return l->vlist[idx]; },
                         [l](uint32_t idx, float sq) { l->cand_dist[idx] = sq; });
        wave_sync();
    }

    // Distance of this lane's slot i of the latest expansion; FLT_MAX where nothing was scored.
    __device__ __forceinline__ float slot_distance(int i) const {
        const float d = finish_row_distance<DIMV>(lds->cand_dist[place[i] & (MAX_CAND - 1)], p.metric);
        return place[i] != kInvalid ? d : FLT_MAX;
    }
    // Buckets of more than 64 slots: from the order of vlist to the slots.  What is not a number is dropped where a beam starts
    // (see absorb) and orders last after that: its bits are above those of infinity.  Returns false if the beam stays as it is;
    // `first` becomes true if the expansion starts a new one.
    __device__ __forceinline__ bool distances_to_slots(bool& first) {
        float d[NC];
#pragma unroll
        for (int i = 0; i < NC; i++) d[i] = slot_distance(i);
        if (first || rank_most == kUnordered) {
            bool some = false, nan = false;
#pragma unroll
            for (int i = 0; i < NC; i++) {
                some |= d[i] < FLT_MAX;
                nan |= d[i] != d[i];
            }
            const uint64_t finite = ballot(some), nans = ballot(nan);
            if (!first && finite == 0) return false;
            first = true;
            rank_most = nans != 0 && finite == 0 ? kUnordered : kRankMost;
            if (finite != 0) {
#pragma unroll
                for (int i = 0; i < NC; i++) {
                    if (d[i] != d[i]) {
                        d[i] = FLT_MAX;
                        lds->cand_id[64 * i + lane] = kInvalid;
                    }
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const uint32_t bits = __float_as_uint(d[i]);
                d[i] = __uint_as_float(bits < 0x7f800000u ? bits : 0x7f800000u);
            }
        }
        wave_sync();
#pragma unroll
        for (int i = 0; i < NC; i++) lds->cand_dist[64 * i + lane] = d[i];
        wave_sync();
        return true;
    }

    // Candidate sort, one network over the wavefront (reference sort_for_candidate, single-warp branch,
    // search_kernel.cuh:9-37): strided load, sort, blocked store of every element.  One candidate slot per lane: `key` is
    // the distance of this lane's slot; `as_is` leaves out the network (see absorb).  What lies behind the slots in use or
    // behind the beam gets an infinite distance, which replaces no beam entry.
    __device__ __forceinline__ void sort_candidates_lane(float key, bool as_is) {
        const uint32_t limit = p.degree < p.beam ? p.degree : p.beam;
        // At most 32 slots in use: the strided load puts them on the even elements of the 64-element network and
        // +inf on the odd ones.  Every comparator of that network then meets at most one real key, or two real
        // keys that the 32-element network compares at the same point of its own sequence and in the same
        // direction, so sorting the 32 slots with the 32-element network gives the same sequence, ties included
        // (the CPU tests compare the two networks on tie-rich inputs), in 15 stages instead of 21.
        // The one exception is a real id whose key is not below FLT_MAX (the build kernels leave the point itself
        // unscored): among the +inf keys its place does depend on the network, so that case takes the long way.
        uint32_t k[1] = {__float_as_uint(key)}, v[1] = {cid};   // few slots: those of the upper half of the wavefront are empty
        if (p.degree <= 32 && ballot(cid != kInvalid && !(key < FLT_MAX)) == 0) {
            KeyNet<32>::sort(k, v, lane);
        } else {
            lds->cand_dist[lane] = key;
            lds->cand_id[lane] = cid;
            wave_sync();
            const uint32_t slot = (lane >> 1) + 32 * (lane & 1);        // reference loads strided: j = lane + 32*i
            k[0] = __float_as_uint(lds->cand_dist[slot]);
            v[0] = lds->cand_id[slot];
            if (!as_is) KeyNet<64>::sort(k, v, lane);
            wave_sync();
        }
        lds->cand_dist[lane] = static_cast<uint32_t>(lane) < limit ? __uint_as_float(k[0]) : __builtin_inff();
        lds->cand_id[lane] = v[0];
        wave_sync();
    }

    // ... with two slots per lane (MAX_CAND == 128)
    __device__ __forceinline__ void sort_candidates_one() {
        float ck[NC];
        uint32_t cv[NC];
#pragma unroll
        for (int r = 0; r < NC; r++) {
            const uint32_t e = NC * lane + r;          // element index in the network
            const uint32_t l32 = e / NC32, i = e % NC32;
            const uint32_t slot = l32 + 32 * i;        // reference loads strided: j = lane + 32*i
            ck[r] = slot < p.degree ? lds->cand_dist[slot] : FLT_MAX;
            cv[r] = slot < p.degree ? lds->cand_id[slot] : kInvalid;
        }
        WaveNet<MAX_CAND>::sort(ck, cv, lane);
        wave_sync();
#pragma unroll
        for (int r = 0; r < NC; r++) {
            const uint32_t e = NC * lane + r;
            lds->cand_dist[e] = ck[r];
            lds->cand_id[e] = cv[r];
        }
        wave_sync();
    }

    // Candidate sort for more than 128 slots (reference two-warp branch, search_kernel.cuh:38-94): the two 32-lane
    // halves of the wavefront are the two warps.  Each sorts its half of the slots, a half-cleaner across the halves
    // leaves the smaller keys with half 0, each half merges.  Only slots below min(degree, beam) are defined afterwards.
    __device__ __forceinline__ void sort_candidates_two() {
        constexpr int PER = MAX_CAND / 2, N = PER / 32;
        const uint32_t w = lane >> 5, l = lane & 31;
        float key[N];
        uint32_t val[N];
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t j = l + 32 * i + PER * w;
            key[i] = j < p.degree ? lds->cand_dist[j] : FLT_MAX;
            val[i] = j < p.degree ? lds->cand_id[j] : kInvalid;
        }
        WaveNet<PER, 32>::sort(key, val, lane);
        wave_sync();
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t jl = N * l + i, j = jl + PER * w;
            if (j < p.degree && jl < p.beam) {
                lds->cand_dist[j] = key[i];
                lds->cand_id[j] = val[i];
            }
        }
        wave_sync();
        const uint32_t warps_used = (p.beam + PER - 1) / PER;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t jl = N * l + i, kl = PER - 1 - jl, j = jl + PER * w, k = MAX_CAND - 1 - j;
            if (w < warps_used && j < p.degree && k < p.degree && kl < p.beam) {
                const float other = lds->cand_dist[k];
                if (key[i] != other && ((w == 0) == (key[i] > other))) {
                    key[i] = other;
                    val[i] = lds->cand_id[k];
                }
            }
        }
        wave_sync();
        WaveNet<PER, 32>::merge(key, val, lane);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t jl = N * l + i, j = jl + PER * w;
            if (w < warps_used && j < p.degree && j < p.beam) {
                lds->cand_dist[j] = key[i];
                lds->cand_id[j] = val[i];
            }
        }
        wave_sync();
    }

    // v of the lane 32 places away: one swap of the 32-lane halves of a register pair and a select
    template <class T>
    static __device__ __forceinline__ T other_half(T v, bool upper) {
        const int x = __builtin_bit_cast(int, v);
        const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);   // s[0]: upper lanes hold the lower half's, s[1]: the reverse
        return __builtin_bit_cast(T, upper ? s[0] : s[1]);
    }

    // Beam merge for a beam of exactly MAX_BEAM entries (beams above 256; the general form follows).  Element
    // NB * lane + r puts the two halves of the beam into the two 32-lane halves of the wavefront, each in the order its
    // merge network wants, so the compare-exchange between the halves is a swap of register halves; and with
    // half == PER the layout [untouched prefix | padding | touched rest] of a half is the half as it stands, whatever
    // the turning points are, so they are not tracked.
    __device__ __forceinline__ void merge_beam_full() {
        bool replaced = false;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t k = MAX_BEAM - 1 - (NB * lane + r);
            if (k < p.degree) {
                const float c = lds->cand_dist[k];
                if (bk[r] > c) {
                    bk[r] = c;
                    bv[r] = lds->cand_id[k];
                    replaced = true;
                }
            }
        }
        if (ballot(replaced) == 0) return;
        const bool upper = lane >= 32;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const float ok = other_half(bk[r], upper);
            const uint32_t ov = other_half(bv[r], upper);
            const bool take = upper ? ok > bk[r] : bk[r] > ok;   // entry j of the first half and entry j of the second change places when the first is larger
            bk[r] = take ? ok : bk[r];
            bv[r] = take ? ov : bv[r];
            __builtin_amdgcn_sched_barrier(0);   // one register at a time: interleaved, the eight exchanges cost the kernel a wavefront per SIMD in registers
        }
        WaveNet<MAX_BEAM / 2, 32>::merge(bk, bv, lane);
    }

    // Beam merge for beams above 256 (reference two-warp branch of sort_for_beam, search_kernel.cuh:149-232), on the beam
    // where it sits; beam a multiple of 16, so that a half is whole lanes.  Half 0 of the beam is in lanes [0, H), half 1
    // in lanes [H, 2H) (H = half / NB), pads behind.  The reference's steps, each of which decides where equal keys end
    // up: candidates displace larger entries from the tail (the smallest touched index of each half, its "turning
    // point", is found with a ballot: indices grow with the lane), the halves are compare-exchanged entry by entry (a
    // lane permutation: same register, lane +-H), each 32-lane half of the wavefront gathers its half of the beam as
    // [untouched prefix | padding | touched rest] -- the source of position q is the same register of another lane,
    // because half and PER - half are multiples of NB -- and merges it, and the beam gathers the results back.  Three
    // lane permutations of the beam's registers; the reference copies the beam through shared memory and finds the
    // turning points with atomics.
    __device__ __forceinline__ void merge_beam_general() {
        constexpr int PER = MAX_BEAM / 2;
        constexpr uint32_t kNone = 0xffffffffu;
        const uint32_t half = p.beam / 2, H = half / NB;
        uint32_t first = kNone;            // this lane's smallest element index that a candidate replaced
#pragma unroll
        for (int r = NB - 1; r >= 0; r--) {
            const uint32_t e = NB * lane + r;
            const uint32_t k = p.beam - 1 - e;
            if (e < p.beam && k < p.degree) {
                const float c = lds->cand_dist[k];
                if (bk[r] > c) {
                    bk[r] = c;
                    bv[r] = lds->cand_id[k];
                    first = e;
                }
            }
        }
        const uint64_t touched = ballot(first != kNone);
        if (touched == 0) return;
        const uint64_t lanes0 = (1ull << H) - 1;
        const uint64_t touched0 = touched & lanes0, touched1 = touched >> H;
        const uint32_t t2 = touched0 ? read_lane(first, __builtin_ctzll(touched0)) : half;
        uint32_t t1 = touched1 ? read_lane(first, static_cast<int>(H) + __builtin_ctzll(touched1)) - half : half;

        // the halves against each other: entry j of half 0 and entry j of half 1 change places when the first is larger
        const bool lower = static_cast<uint32_t>(lane) < H, upper = !lower && static_cast<uint32_t>(lane) < 2 * H;
        const int partner = lower ? lane + static_cast<int>(H) : (upper ? lane - static_cast<int>(H) : lane);
        uint32_t moved = kNone;
#pragma unroll
        for (int r = NB - 1; r >= 0; r--) {
            const float ok = shfl_f32(bk[r], partner);
            const uint32_t ov = shfl_u32(bv[r], partner);
            const bool take = lower ? bk[r] > ok : (upper && ok > bk[r]);
            if (take && lower) moved = NB * lane + r;
            bk[r] = take ? ok : bk[r];
            bv[r] = take ? ov : bv[r];
            __builtin_amdgcn_sched_barrier(0);   // one register at a time (interleaved, the permutations of a step hold the beam twice)
        }
        const uint64_t movers = ballot(moved != kNone);
        const uint32_t t0 = movers ? read_lane(moved, __builtin_ctzll(movers)) : half;
        if (t2 < half) t1 = t2;

        // each 32-lane half gathers its half of the beam as [untouched prefix | padding | touched rest]; register i of a
        // position comes from register i of another lane, so the beam's registers are rewritten in place
        const uint32_t w = static_cast<uint32_t>(lane) >> 5, l = static_cast<uint32_t>(lane) & 31;
        const uint32_t turning = w ? t1 : t0;
        const uint32_t gap = PER - half;                       // the rest sits `gap` positions further on
        const int from_prefix = static_cast<int>(l + H * w), from_rest = static_cast<int>(l + H * w) - static_cast<int>(gap / NB);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const uint32_t q = NB * l + i;
            const bool in_prefix = q < turning;
            const bool in_rest = q >= gap && q - gap >= turning;     // q - gap < half holds for every q < PER
            const int src = in_prefix ? from_prefix : (in_rest ? from_rest : lane);
            const float k = shfl_f32(bk[i], src);
            const uint32_t v = shfl_u32(bv[i], src);
            bk[i] = in_prefix || in_rest ? k : FLT_MAX;
            bv[i] = in_prefix || in_rest ? v : kInvalid;
            __builtin_amdgcn_sched_barrier(0);
        }
        WaveNet<PER, 32>::merge(bk, bv, lane);
        // back into beam order: the first `half` positions of half-wave w are elements [half * w, half * w + half)
        const uint32_t w2 = static_cast<uint32_t>(lane) >= H ? 1u : 0u;
        const int back = static_cast<int>(static_cast<uint32_t>(lane) - H * w2 + 32 * w2) & 63;
        const bool live = static_cast<uint32_t>(lane) < 2 * H;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const float k = shfl_f32(bk[r], back);
            const uint32_t v = shfl_u32(bv[r], back);
            bk[r] = live ? k : FLT_MAX;
            bv[r] = live ? v : kInvalid;
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // The last beam entry's key, as bits.
    __device__ __forceinline__ uint32_t tail_key() const {
        // The beam is ascending, so its last entry is the largest key of the lane that holds it among that lane's entries
        // below `beam` (written as a maximum: a chain of selects between the registers becomes a run-time index, which
        // moves the beam out of the registers).  Keys are not negative, so they compare as their bits; what is not a number is
        // above everything else and enters nowhere.
        uint32_t tail;
        if (p.beam % NB == 0) {   // the last entry is the last register of a lane (beams are multiples of 32 as a rule)
            tail = read_lane(__float_as_uint(bk[NB - 1]), static_cast<int>(p.beam / NB) - 1);
        } else {
            const uint32_t last = p.beam - 1;
            uint32_t mine = __float_as_uint(bk[0]);
#pragma unroll
            for (int r = 1; r < NB; r++) {
                const uint32_t k = NB * lane + r <= static_cast<int>(last) ? __float_as_uint(bk[r]) : 0u;
                mine = mine > k ? mine : k;
            }
            tail = read_lane(mine, static_cast<int>(last / NB));
        }
        return tail;
    }

    // The candidates of the latest expansion that are below the last beam entry, as a lane mask (one candidate slot per
    // lane).  None: the beam stays as it is -- the half-cleaner of the merge replaces an entry only by a strictly smaller
    // candidate, entry `beam - 1 - k` by the k-th smallest, so if even the smallest candidate is not below the largest
    // entry nothing is replaced, and the candidate sort in front of it only feeds that test.  Half of all iterations of
    // a wide beam end here (the further a search has come, the fewer neighbours of its frontier are nearer than the worst
    // entry it holds), for one comparison per lane.
    __device__ __forceinline__ uint64_t entering(float ck) const {
        static_assert(MAX_CAND == 64, "one candidate slot per lane");
        const uint32_t tail = tail_key();
        return ballot(__float_as_uint(ck) < tail);
    }

    // Beam merge for beams of up to 256 entries (reference sort_for_beam, single-warp branch): the k-th smallest candidate
    // displaces entry MAX_BEAM - 1 - k if that is larger, then the merge network runs.
    __device__ __forceinline__ void merge_beam() {
        bool replaced = false;
        uint32_t k[NB];
#pragma unroll
        for (int r = 0; r < NB; r++) k[r] = __float_as_uint(bk[r]);
        if constexpr (NC == 1) {
            // a lane's candidates are NB neighbouring places, in reverse; behind those that count the distance is infinite
            struct alignas(4 * NB) Keys { float d[NB]; };
            struct alignas(4 * NB) Ids { uint32_t id[NB]; };
            const int from = NB * (63 - lane);
            if (from < MAX_CAND) {
                const Keys c = *reinterpret_cast<const Keys*>(lds->cand_dist + from);
                const Ids ci = *reinterpret_cast<const Ids*>(lds->cand_id + from);
#pragma unroll
                for (int r = 0; r < NB; r++) {
                    const uint32_t o = __float_as_uint(c.d[NB - 1 - r]);
                    const bool smaller = o < k[r];
                    bv[r] = smaller ? ci.id[NB - 1 - r] : bv[r];
                    k[r] = smaller ? o : k[r];
                    replaced |= smaller;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const uint32_t e = NB * lane + r;
                const uint32_t j = MAX_BEAM - 1 - e;
                if (j < p.beam && j < p.degree) {
                    const uint32_t c = __float_as_uint(lds->cand_dist[j]);
                    if (k[r] > c) {
                        k[r] = c;
                        bv[r] = lds->cand_id[j];
                        replaced = true;
                    }
                }
            }
        }
        // Nothing replaced: the beam is still the ascending sequence the previous merge left, and the merge
        // network (strict comparisons) is the identity on it.
        if (ballot(replaced) == 0) return;
        KeyNet<MAX_BEAM>::merge(k, bv, lane);
#pragma unroll
        for (int r = 0; r < NB; r++) bk[r] = __uint_as_float(k[r]);
        reset_pads();
    }

    // entries pushed past the end of the beam
    __device__ __forceinline__ void reset_pads() {
        if (p.beam == MAX_BEAM) return;   // a beam that fills its bucket has nothing behind it (and the lane masks of this loop are not held)
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t e = NB * lane + r;
            if (e >= p.beam) {
                bk[r] = FLT_MAX;
                bv[r] = kInvalid;
            }
        }
    }

    // ---- few candidates below the last beam entry --------------------------------------------------------------------
    // Where all keys involved are distinct there is one ascending order, whatever network makes it.  Then up to kInsertMost
    // candidates are inserted one by one: with the beam ascending, entry e becomes the median of entry e - 1, the candidate
    // and itself.  That is 4 NB + 5 vector instructions a candidate, and no LDS, against the candidate sort (70) and the
    // beam merge (27 / 55 / 116 for NB = 1 / 2 / 4) of the general way.  Where keys are equal the networks decide the order
    // (the reference's comparators), so an equal pair within the beam (`tied`, kept since the last merge: insertions make
    // none) or with a candidate sends the expansion there.  Integer rows meet equal distances often in wide beams, float
    // rows next to never.
    static constexpr uint32_t kInsertMost = 8;
    // Up to kRankMost candidates that differ from each other are ranked by counting (4 instructions each), more are sorted.
    // A beam that starts with rows at an infinite distance has all of them sorted: the empty slots of the sorted list, left out
    // of the ranked one, displace such rows, which only come in at the start.
    static constexpr int kRankMost = 14;

    // whether two beam entries have equal keys, or an entry orders like the padding without being padding
    __device__ __forceinline__ bool has_ties() const {
        uint64_t any = 0;
        const uint32_t pad = __float_as_uint(FLT_MAX);
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t k = __float_as_uint(bk[r]);
            const uint32_t next = r + 1 < NB ? __float_as_uint(bk[r + 1 < NB ? r + 1 : 0])
                                             : static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(__float_as_uint(bk[0])), 0x130, 0xf, 0xf, false));   // wave_shl:1
            const uint64_t real = ballot(k < pad);
            any |= (ballot(k == next) & real) | (ballot(bv[r] != kInvalid) & ~real);
        }
        return any != 0;
    }
    __device__ __forceinline__ bool meets_equal(float key, uint64_t em) const {
        uint64_t equal = 0;
        for (uint64_t rest = em; rest; rest &= rest - 1) {
            const int j = __builtin_ctzll(rest);
            const float c = read_lane(key, j);
            equal |= ballot(key == c) & (rest & (rest - 1));   // a later candidate with this key
#pragma unroll
            for (int r = 0; r < NB; r++) equal |= ballot(bk[r] == c);
        }
        return equal != 0;
    }
    // the value one lane below (lane 0: zero)
    template <class T>
    static __device__ __forceinline__ T lane_below(T x) {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true));   // wave_shr:1
    }
    __device__ __forceinline__ void insert(float key, uint64_t em) {
        for (uint64_t rest = em; rest; rest &= rest - 1) {
            const int j = __builtin_ctzll(rest);
            const float c = read_lane(key, j);
            const uint32_t id = read_lane(cid, j);
            const float pk = lane_below(bk[NB - 1]);
            const uint32_t pv = lane_below(bv[NB - 1]);
            uint64_t below[NB];   // lanes whose entry r comes behind the candidate
#pragma unroll
            for (int r = 0; r < NB; r++) below[r] = ballot(c < bk[r]);
            const uint64_t below_first = below[NB - 1] << 1;   // ... whose entry -1, the last one of the lane below, does
#pragma unroll
            for (int r = NB - 1; r >= 0; r--) {
                const float prev_k = r ? bk[r ? r - 1 : 0] : pk;
                const uint32_t prev_v = r ? bv[r ? r - 1 : 0] : pv;
                const uint64_t prev_below = r ? below[r ? r - 1 : 0] : below_first;
                bk[r] = __builtin_amdgcn_fmed3f(prev_k, c, bk[r]);
                bv[r] = select_by_mask(bv[r], select_by_mask(id, prev_v, prev_below), below[r]);
            }
        }
        reset_pads();
    }
    // The entering candidates in ascending order at the front of the candidate lists; false if two have the same key.
    __device__ __forceinline__ bool rank_candidates(float key, uint64_t em) {
        uint32_t rank = 0;
        uint64_t equal = 0;
        for (uint64_t rest = em; rest; rest &= rest - 1) {
            const float c = read_lane(key, __builtin_ctzll(rest));
            equal |= ballot(key == c) & (rest & (rest - 1));
            rank += c < key ? 1u : 0u;
        }
        if (equal != 0) return false;
        lds->cand_dist[lane] = __builtin_inff();
        wave_sync();
        if (((em >> lane) & 1) != 0 && rank < p.beam) {
            lds->cand_dist[rank] = key;
            lds->cand_id[rank] = cid;
        }
        wave_sync();
        return true;
    }

    // What the first candidates of a beam say about it; beside rows at a finite distance those at none are dropped.
    __device__ __forceinline__ void start_beam(float& key) {
        const uint64_t finite = ballot(key < FLT_MAX), nans = ballot(key != key);
        rank_most = finite == 0 && nans != 0 ? kUnordered : ballot(key > FLT_MAX) != 0 ? 0 : kRankMost;
        if (finite != 0 && key != key) {
            key = FLT_MAX;
            cid = kInvalid;
        }
    }

    // reference update_result_buffer: sort the candidates, then fold them into the beam
    //
    // Rows at a distance that is not a number (a NaN in the row or in the query) compare with nothing, and a network that
    // meets one leaves its other keys unsorted.  They are no candidates, except while there are no others: the entry's
    // neighbours then make up the beam unsorted and are expanded like any entry (a query with a NaN ends with them), until an
    // expansion finds a row at a finite distance and a new beam starts with that expansion's candidates.
    __device__ __forceinline__ void absorb(bool first, row_data<DIMV> data) {
        // No row scored: every candidate distance is FLT_MAX, the sort would not move anything (equal keys are never
        // exchanged) and no candidate can displace a beam entry, so the beam stays as it is.
        if (!first && last_scored == 0) return;
        if constexpr (NC == 1) {
            float key = slot_distance(0);
            if (first) {
                start_beam(key);
                wave_sync();
                sort_candidates_lane(key, rank_most == kUnordered);
            } else {
                const uint64_t em = entering(key);
                if (em == 0) return;
                const uint32_t m = __popcll(em);
                if (m <= kInsertMost && !tied && !meets_equal(key, em)) {
                    insert(key, em);
                    return;
                }
                wave_sync();
                if (static_cast<int>(m) > rank_most || !rank_candidates(key, em)) {
                    if constexpr (ROUGH) {   // the networks decide between equal keys by where all the others are
                        if (passed_over != 0) {
                            measure(passed_over, data);
                            key = slot_distance(0);
                        }
                    }
                    // An unordered beam's keys are above all others and count as tied, so every candidate that enters one comes here
                    // (one that took none of its rows in has none to expand either, and no candidates follow).
                    if (rank_most == kUnordered) {
                        if (ballot(key < FLT_MAX) == 0) return;
                        start_beam(key);
                        first = true;
                    }
                    sort_candidates_lane(key, false);
                }
            }
        } else {
            if (!distances_to_slots(first)) return;
            if constexpr (MAX_CAND > 128) sort_candidates_two();
            else sort_candidates_one();
        }
        if (first) {
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const uint32_t e = NB * lane + r;
                const bool take = e < p.beam && e < p.degree;
                bk[r] = take ? lds->cand_dist[e] : FLT_MAX;
                bv[r] = take ? lds->cand_id[e] : kInvalid;
            }
        } else if constexpr (MAX_BEAM > 256) {
            if constexpr (WHOLE) merge_beam_full();
            else merge_beam_general();
        } else {
            merge_beam();
        }
        wave_sync();
        if constexpr (NC == 1) tied = has_ties();
    }

    // first unexplored beam entry (reference select_current_point); marks it explored
    __device__ __forceinline__ uint32_t select_parent() {
        // Entries behind the beam are pads (kInvalid), which carry the explored bit like every unfilled entry.  One compare
        // per register; the rest is scalar, and the chosen entry is read by its lane number and marked under a one-lane mask.
        uint64_t open[NB], any = 0;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            open[r] = ballot(static_cast<int>(bv[r]) >= 0);
            any |= open[r];
        }
        if (any == 0) return kInvalid;
        const int src = __builtin_ctzll(any);
        uint32_t mine = 0;
        bool taken = false;
#pragma unroll
        for (int r = 0; r < NB; r++) {
            if (!taken && ((open[r] >> src) & 1) != 0) {
                mine = read_lane(bv[r], src);
                bv[r] = select_by_mask(bv[r], bv[r] | kExplored, 1ull << src);
                taken = true;
            }
        }
        return mine;
    }

    __device__ __forceinline__ void restore_hash() {
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const uint32_t e = NB * lane + r;
            if (e < p.beam) hash_insert(hash, p.hash_bit, bv[r] & kClean);
        }
    }

    // main loop; candidates of the entry expansion must already be in LDS
    __device__ __forceinline__ void run(const uint32_t* graph, row_data<DIMV> data, uint32_t self_id) {
        uint32_t iter = 0;
        bool terminate = false;
        while (true) {
            asm volatile("" : "+v"(lane));   // a dozen addresses and masks made from the lane number are cheaper made anew in an iteration than held (and spilled) across it
            absorb(iter == 0, data);
            cnt.iterations++;
            const bool reset_now = count_down();
            if (reset_now) {
                hash_clear(hash, p.hash_bit, lane);
                wave_sync();
            }
            if (iter + 1 == p.max_iterations) break;
            const uint32_t parent = select_parent();
            if (parent == kInvalid) terminate = true;
            if (reset_now) {
                restore_hash();
                wave_sync();
            }
            if (terminate && iter >= p.min_iterations) break;
            expand(parent, graph, data, self_id, kInvalid, false);
            iter++;
        }
    }

    // `counters` holds kCounterStripes x 3 u64 (striped by workgroup: a single shared address would serialise the
    // whole launch); the host adds the stripes up
    __device__ __forceinline__ void flush_counters(unsigned long long* counters) {
        if (counters != nullptr && lane == 0) {
            unsigned long long* slot = counters + 3 * (blockIdx.x % kCounterStripes);
            atomicAdd(&slot[0], static_cast<unsigned long long>(cnt.iterations));
            atomicAdd(&slot[1], static_cast<unsigned long long>(cnt.rows_scored));
            atomicAdd(&slot[2], static_cast<unsigned long long>(cnt.graph_rows));
        }
    }
};

// Nearest centroid by the reference's sort network (search_kernel.cuh:259-268, distance.cuh:29-60):
// strided load, blocked store, element 0 is the winner.  One wavefront; scratch holds `centroid_num` pairs.
template <int MAX_CENTROID, int DIMV, bool TEAM = false>
__device__ __forceinline__ uint32_t nearest_centroid(const RowRegs<DIMV>& q, const float* centroids, uint32_t centroid_num,
                                                     uint32_t dim, int metric, float* cent_dist, int lane) {
    using Shape = RowShape<DIMV>;
    const int g = Shape::row_of_lane(lane), t = Shape::lane_in_row(lane);
    for (uint32_t c0 = 0; c0 < centroid_num; c0 += Shape::ROWS) {
        const uint32_t c = c0 + g;
        RowRegs<DIMV> row;
        if (c < centroid_num) {
            load_row<DIMV>(row, centroids + static_cast<size_t>(c) * dim, dim, t);
        } else {
            row = q;
        }
        const float d = finish_distance(row_sum<DIMV>(partial_sqdist<DIMV>(q, row)), metric);
        if (t == 0 && c < centroid_num) cent_dist[c] = d;
    }
    wave_sync_in<TEAM>();
    constexpr int NR = KeyNet<MAX_CENTROID>::NR;
    constexpr int N32 = MAX_CENTROID / 32;
    uint32_t k[NR], v[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const uint32_t e = NR * lane + r;
        const uint32_t j = (e / N32) + 32 * (e % N32);
        const bool ok = (MAX_CENTROID >= 64 || lane < 32) && j < centroid_num;
        k[r] = __float_as_uint(ok ? cent_dist[j] : FLT_MAX);
        v[r] = ok ? j : kInvalid;
    }
    KeyNet<MAX_CENTROID>::sort(k, v, lane);
    wave_sync_in<TEAM>();
    const uint32_t nearest = read_lane(v[0], 0);
    return nearest == kInvalid ? 0u : nearest;   // nothing below the padding: a query with a NaN
}

}  // namespace glide
