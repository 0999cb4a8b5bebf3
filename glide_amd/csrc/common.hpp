// Wave64 device primitives shared by every GLIDE kernel on gfx950 (CDNA4).
//
// One wavefront = 64 lanes.  All per-item kernels (search, sub-graph build, refine) give one item to one
// wavefront, so the "warp 0 / other warps" split and the block barriers of the reference collapse into
// straight-line wave code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>

namespace glide {

constexpr uint32_t kInvalid = 0xffffffffu;
constexpr uint32_t kExplored = 0x80000000u;  // reference utils.cuh:5-8
constexpr uint32_t kClean = 0x7fffffffu;
constexpr int kWave = 64;

enum Metric : int { kEuclidean = 0, kCosine = 1 };  // reference params.cuh:5-8

__host__ __device__ constexpr uint32_t round_up32(uint32_t p) { return (p + 31u) & ~31u; }  // utils.cuh:21-23
// a / b rounded up, without the wrap of (a + b - 1) when a is within b of 2^32
__host__ __device__ constexpr uint32_t ceil_div(uint32_t a, uint32_t b) { return a / b + (a % b != 0); }

__device__ __forceinline__ int lane_id() { return static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u))); }

// ---------------------------------------------------------------- cross-lane exchange, compile-time xor mask
// xor 1,2: DPP quad_perm; xor 4: two banked DPP row shifts; xor 8: DPP row_ror:8; xor 16: ds_swizzle (LDS
// crossbar, no memory); xor 32: ds_bpermute.
template <int MASK>
__device__ __forceinline__ int lane_xor_i(int v) {
    static_assert(MASK == 1 || MASK == 2 || MASK == 4 || MASK == 8 || MASK == 16 || MASK == 32, "xor mask");
    // mov_dpp leaves the destination's previous value undefined for lanes the pattern does not write; every pattern
    // below writes all 64 lanes, so no register has to be initialised first
    if constexpr (MASK == 1) {
        return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, false);  // quad_perm:[1,0,3,2]
    } else if constexpr (MASK == 2) {
        return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, false);  // quad_perm:[2,3,0,1]
    } else if constexpr (MASK == 4) {
        int r = __builtin_amdgcn_mov_dpp(v, 0x104, 0xf, 0x5, false);    // row_shl:4 -> banks 0,2 read lane+4
        r = __builtin_amdgcn_update_dpp(r, v, 0x114, 0xf, 0xA, false);  // row_shr:4 -> banks 1,3 read lane-4
        return r;
    } else if constexpr (MASK == 8) {
        return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, false);  // row_ror:8
    } else if constexpr (MASK == 16) {
        return __builtin_amdgcn_ds_swizzle(v, 0x401F);  // BITMODE and=0x1f or=0 xor=0x10
    } else {
        return __builtin_amdgcn_ds_bpermute((lane_id() ^ 32) << 2, v);
    }
}
// A 64-lane predicate mask with every bit moved to the lane MASK away (the partner's predicate), on the scalar unit.
template <int MASK>
__device__ __forceinline__ uint64_t mask_xor(uint64_t m) {
    constexpr uint64_t low = MASK == 1 ? 0x5555555555555555ull : MASK == 2 ? 0x3333333333333333ull : MASK == 4 ? 0x0F0F0F0F0F0F0F0Full
                           : MASK == 8 ? 0x00FF00FF00FF00FFull : MASK == 16 ? 0x0000FFFF0000FFFFull : 0x00000000FFFFFFFFull;
    return ((m & low) << MASK) | ((m >> MASK) & low);
}
// per-lane select driven by a scalar 64-bit mask: lane l gets `b` where bit l is set, else `a`
__device__ __forceinline__ float select_by_mask(float a, float b, uint64_t mask) {
    float out;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(out) : "v"(a), "v"(b), "s"(mask));
    return out;
}
__device__ __forceinline__ uint32_t select_by_mask(uint32_t a, uint32_t b, uint64_t mask) {
    uint32_t out;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(out) : "v"(a), "v"(b), "s"(mask));
    return out;
}
template <int MASK>
__device__ __forceinline__ float lane_xor(float v) { return __builtin_bit_cast(float, lane_xor_i<MASK>(__builtin_bit_cast(int, v))); }
template <int MASK>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) { return static_cast<uint32_t>(lane_xor_i<MASK>(static_cast<int>(v))); }

__device__ __forceinline__ float read_lane(float v, int lane) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane)); }
__device__ __forceinline__ uint32_t read_lane(uint32_t v, int lane) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane)); }
__device__ __forceinline__ uint32_t shfl_u32(uint32_t v, int src_lane) { return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(src_lane << 2, static_cast<int>(v))); }
__device__ __forceinline__ float shfl_f32(float v, int src_lane) { return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src_lane << 2, __builtin_bit_cast(int, v))); }

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }
// number of set bits of `mask` strictly below this lane
__device__ __forceinline__ uint32_t prefix_count(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// Sum over each 32-lane half of the wave; every lane of a half ends with that half's total.
__device__ __forceinline__ float half_wave_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false));  // row_half_mirror
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, false));  // row_mirror
    v += lane_xor<16>(v);
    return v;
}
// Sum over the whole wave; every lane ends with the total.
__device__ __forceinline__ float wave_sum(float v) {
    v = half_wave_sum(v);
    v += lane_xor<32>(v);
    return v;
}

// Prefix sum over the 64 lanes without LDS traffic: four shifted adds inside each row of 16 lanes, then lane 15 of a row
// is added to the next row (rows 1 and 3) and lane 31 to the upper half (rows 2 and 3).  Lanes a step does not feed add 0.
__device__ __forceinline__ uint32_t wave_exclusive_scan(uint32_t value, uint32_t& total) {
    int x = static_cast<int>(value);
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);   // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);   // row_bcast:31
    total = static_cast<uint32_t>(__builtin_amdgcn_readlane(x, 63));
    return static_cast<uint32_t>(x) - value;
}

// ---------------------------------------------------------------- LDS open-addressing hash set (reference hashmap.cuh:23-56)
__device__ __forceinline__ void hash_clear(uint32_t* table, uint32_t bitlen, int lane) {
    if (bitlen >= 8) {   // 16 bytes a lane (the tables of the beam kernels are 16-byte aligned)
        const uint4 none = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
        for (uint32_t i = lane; i < (1u << (bitlen - 2)); i += kWave) reinterpret_cast<uint4*>(table)[i] = none;
        return;
    }
    for (uint32_t i = lane; i < (1u << bitlen); i += kWave) table[i] = kInvalid;
}
// returns 1 iff `key` was newly stored; 0 if present or the table is full.  One exit, the outcome read off the last slot
// afterwards (a loop with three outcomes costs twice the mask bookkeeping per probe, and so does an outcome that the loop
// carries along as a mask: hence the opaque copy).  Four vector instructions a probe: the slot is a byte offset, wrapped by a
// mask, and the count of probes is the same in every lane still probing, so it is kept on the scalar unit.  An expansion
// probes four times or so, restoring a beam after a reset as often for each of its registers: with eight instructions a probe
// they were a fifth of what a beam search issues.
__device__ __forceinline__ uint32_t hash_insert(uint32_t* table, uint32_t bitlen, uint32_t key) {
    const uint32_t mask = (4u << bitlen) - 4u;
    uint32_t at = ((key ^ (key >> bitlen)) << 2) & mask, left = 1u << bitlen, old;
    do {
        old = atomicCAS(reinterpret_cast<uint32_t*>(reinterpret_cast<unsigned char*>(table) + at), kInvalid, key);
        at = (at + 4u) & mask;
        left = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(left))) - 1u;
    } while ((old != kInvalid) & (old != key) & (left != 0));
    asm("" : "+v"(old));
    return old == kInvalid ? 1u : 0u;
}

// ---------------------------------------------------------------- row distance, several rows per wave-wide load
// A row is read by a group of LPR adjacent lanes, 16 bytes per lane and load, NV loads per lane; lane t of a group
// owns dims [(c*LPR + t)*4, +4) of load c, so one load instruction touches LPR*16 contiguous bytes of each row.
// Narrow rows use narrow groups: the cross-lane sum then needs log2(LPR) steps instead of 5 and one instruction
// serves 64/LPR rows.  DIMV selects the shape by row length (dim <= 128*DIMV):
//   DIMV 1: 8 lanes x 4 loads (8 rows per wavefront)    DIMV 2: 16 lanes x 4 loads (4 rows)
//   DIMV 4: 32 lanes x 4 loads (2 rows)                 DIMV 8 / 16: 32 lanes x 8 / 16 loads (2 rows)
//   DIMV 32: 64 lanes x 16 loads (1 row; up to 4096 dims)
//   DIMV -1: rows of bytes, 8 lanes x 1 load (8 rows, up to 128 dims)    DIMV -2: 16 lanes x 1 load (4 rows, up to 256 dims)
template <int DIMV>
struct RowShape {
    static_assert(DIMV == 1 || DIMV == 2 || DIMV == 4 || DIMV == 8 || DIMV == 16 || DIMV == 32 || DIMV == -1 || DIMV == -2, "row shape");
    static constexpr bool BYTES = DIMV < 0;
    static constexpr int LPR = DIMV == 1 || DIMV == -1 ? 8 : (DIMV == 2 || DIMV == -2 ? 16 : (DIMV == 32 ? 64 : 32));
    static constexpr int NV = BYTES ? 1 : DIMV >= 16 ? 16 : (DIMV == 8 ? 8 : 4);
    static constexpr int ROWS = 64 / LPR;
    static constexpr int STRIDE = LPR * 16;   // bytes from row to row, where rows are bytes
    static __device__ __forceinline__ int lane_in_row(int lane) { return lane & (LPR - 1); }
    static __device__ __forceinline__ int row_of_lane(int lane) { return lane / LPR; }
};

// Rows of whole numbers 0 .. 255 (image descriptors, quantised embeddings) are searched as bytes: a quarter of the memory
// traffic, and |x - q|^2 = x.x - 2 x.q + q.q takes eight dot products of four bytes for sixteen dims in place of 32 fp32
// instructions.  All of it is integer arithmetic and exact; with at most kMostByteDims dims every sum the fp32 form makes
// stays below 2^24 and is exact as well, so both give the same distances to the bit.  Measured on 128 dims, fp32 : bytes:
// 10 000 searches of a million rows at beam 64 1 347 : 479 us (rows from memory; 1 query 124 : 108), at beam 256 on the mixture,
// whose rows come from the caches, 2 320 : 1 600; refinement of a million points 71 : 52 ms (0.95 of the vector issue rate),
// sub-graphs 44 : 31 ms.
constexpr uint32_t kMostByteDims = 256;   // 256 * 255^2 < 2^24
constexpr uint32_t kMostByteDegree = 64;  // the searches over rows of bytes are built for one candidate slot a lane

// a lane's share of a row
template <int DIMV, bool BYTES = RowShape<DIMV>::BYTES>
struct RowRegs {
    float4 v[RowShape<DIMV>::NV];
};
template <int DIMV>
struct RowRegs<DIMV, true> {
    uint4 v;
    uint32_t sq;   // the share's own squared length: set where the row is what others are measured against
};

template <bool BYTES> struct RowData { using type = const float*; };
template <> struct RowData<true> { using type = const unsigned char*; };
template <int DIMV>
using row_data = typename RowData<RowShape<DIMV>::BYTES>::type;   // where rows are read from

template <int DIMV>
__device__ __forceinline__ row_data<DIMV> row_at(row_data<DIMV> rows, uint32_t id, uint32_t dim) {
    if constexpr (RowShape<DIMV>::BYTES) return rows + static_cast<size_t>(id) * RowShape<DIMV>::STRIDE;
    else return rows + static_cast<size_t>(id) * dim;
}

// t = RowShape<DIMV>::lane_in_row(lane)
template <int DIMV, bool FULL = false>   // FULL: dim fills the shape exactly (rows of bytes always do: zeros behind them)
__device__ __forceinline__ void load_row(RowRegs<DIMV>& r, row_data<DIMV> row, uint32_t dim, int t) {
    if constexpr (RowShape<DIMV>::BYTES) {
        r.v = *reinterpret_cast<const uint4*>(row + t * 16);
    } else {
#pragma unroll
        for (int c = 0; c < RowShape<DIMV>::NV; c++) {
            const uint32_t d0 = (c * RowShape<DIMV>::LPR + t) * 4;
            r.v[c] = FULL || d0 < dim ? *reinterpret_cast<const float4*>(row + d0) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
}

__device__ __forceinline__ uint32_t dot_bytes(const uint4& a, const uint4& b, uint32_t acc) {
    acc = __builtin_amdgcn_udot4(a.x, b.x, acc, false);
    acc = __builtin_amdgcn_udot4(a.y, b.y, acc, false);
    acc = __builtin_amdgcn_udot4(a.z, b.z, acc, false);
    return __builtin_amdgcn_udot4(a.w, b.w, acc, false);
}
// a row that others are measured against
template <int DIMV>
__device__ __forceinline__ void load_reference(RowRegs<DIMV>& r, row_data<DIMV> row, uint32_t dim, int t) {
    load_row<DIMV>(r, row, dim, t);
    if constexpr (RowShape<DIMV>::BYTES) r.sq = dot_bytes(r.v, r.v, 0u);
}

// Sixteen fp32 values from `row + first` on as bytes; values behind `dim` are zeros.  False: one is no whole number 0 .. 255.
__device__ __forceinline__ bool pack_bytes(const float* row, uint32_t first, uint32_t dim, uint4& out) {
    uint32_t word[4];
    bool exact = true;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const uint32_t d0 = first + 4 * w;
        const float4 x = d0 < dim ? *reinterpret_cast<const float4*>(row + d0) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float v[4] = {x.x, x.y, x.z, x.w};
        word[w] = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool in_range = v[e] >= 0.f && v[e] <= 255.f;   // false for what is not a number
            const uint32_t b = in_range ? static_cast<uint32_t>(v[e]) : 0u;
            exact &= in_range && static_cast<float>(b) == v[e];
            word[w] |= b << (8 * e);
        }
    }
    out = make_uint4(word[0], word[1], word[2], word[3]);
    return exact;
}

__device__ __forceinline__ float sqdist4(const float4& a, const float4& b, float acc) {
    const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z, dw = a.w - b.w;
    acc = fmaf(dx, dx, acc);
    acc = fmaf(dy, dy, acc);
    acc = fmaf(dz, dz, acc);
    acc = fmaf(dw, dw, acc);
    return acc;
}

template <int DIMV>
__device__ __forceinline__ float partial_sqdist(const RowRegs<DIMV>& a, const RowRegs<DIMV>& b) {
    float acc = 0.f;
#pragma unroll
    for (int c = 0; c < RowShape<DIMV>::NV; c++) acc = sqdist4(a.v[c], b.v[c], acc);
    return acc;
}

// ---------------------------------------------------------------- fp32 rows, a first look in fp16
// Nine of ten rows that a search scores come in no nearer than the worst entry it holds, and of them only that much has to be
// known.  A copy of the rows in fp16, scaled by one power of two for all of them, says it from half the bytes and half the
// instructions (a packed difference and a dot product for two values, in place of four): with s the distance of the rounded rows,
// the distance as the exact pass would compute it lies in [rough_least, rough_most].  Rounding moves a row x by at most
// r |x| + t (t: sqrt(dim) times the smallest normal fp16 number, whatever becomes of the numbers below it; r <= 2^-11, measured
// over the rows when they are packed: some 0.4 of that), the reference q likewise, |x| <= |q| + |q - x|; the differences are off
// by 2^-11 of themselves or t, and the sums of either pass by (dim + 8) 2^-24 of themselves (`slack` is four times that).  What the
// bounds leave open is measured exactly, so nothing but the traffic changes.
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
struct RoughRows {
    const _Float16* rows;   // num x stride, zeros behind a row's dims
    uint32_t stride;
    float unit;             // what a value of 1 stands for; NaN where some value is infinite or none: then nothing is decided
    float turn;             // r
    float tiny;             // 3 t
    float slack;
};
template <int DIMV>
struct RoughRegs {          // a lane's share of such a row: 8 (c LPR + t) .. + 7 for the c-th
    static constexpr int NV = RowShape<DIMV>::NV / 2;
    uint4 v[NV];
};
constexpr uint32_t kRoughHeader = 256;   // bytes before the rows: the largest |value| and r, as bits
inline __host__ __device__ uint32_t rough_stride(uint32_t dim) { return (dim + 7) & ~7u; }
// The largest value comes to lie in [2^13, 2^14): differences of two stay in range.
__device__ __forceinline__ float rough_unit(uint32_t max_bits) {
    if (max_bits >= 0x7f800000u) return __builtin_nanf("");
    const uint32_t e = max_bits >> 23;
    return __uint_as_float((e < 14u ? 1u : e - 13u) << 23);
}
__device__ __forceinline__ RoughRows rough_rows(const unsigned char* held, uint32_t dim) {
    RoughRows r;
    r.rows = reinterpret_cast<const _Float16*>(held + kRoughHeader);
    r.stride = rough_stride(dim);
    r.unit = rough_unit(*reinterpret_cast<const uint32_t*>(held));
    r.turn = __uint_as_float(reinterpret_cast<const uint32_t*>(held)[1]);
    r.tiny = sqrtf(static_cast<float>(dim)) * 3 * 6.2e-5f * r.unit;
    r.slack = static_cast<float>(dim + 8) * 2.4e-7f;
    return r;
}
template <int DIMV, bool FULL>
__device__ __forceinline__ void load_rough(RoughRegs<DIMV>& regs, const RoughRows& r, uint32_t id, uint32_t dim, int t) {
    const _Float16* row = r.rows + static_cast<size_t>(id) * r.stride;
#pragma unroll
    for (int c = 0; c < RoughRegs<DIMV>::NV; c++) {
        const uint32_t d0 = (c * RowShape<DIMV>::LPR + t) * 8;
        regs.v[c] = FULL || d0 < dim ? *reinterpret_cast<const uint4*>(row + d0) : make_uint4(0u, 0u, 0u, 0u);
    }
}
// a lane's part of the squared distance, in units
template <int DIMV>
__device__ __forceinline__ float rough_sqdist(const RoughRegs<DIMV>& a, const RoughRegs<DIMV>& b) {
    float acc[4] = {};   // four chains: a product is not ready for the next instruction
#pragma unroll
    for (int c = 0; c < RoughRegs<DIMV>::NV; c++) {
        const uint32_t of_a[4] = {a.v[c].x, a.v[c].y, a.v[c].z, a.v[c].w}, of_b[4] = {b.v[c].x, b.v[c].y, b.v[c].z, b.v[c].w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const half2v d = __builtin_bit_cast(half2v, of_a[e]) - __builtin_bit_cast(half2v, of_b[e]);
            acc[e] = __builtin_amdgcn_fdot2(d, d, acc[e], false);
        }
    }
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}
constexpr float kRoughTurn = 4.93e-4f;   // 2^-11 and a little, the most that r is
// sq: squared distance of the rounded rows; norm: the reference's length, or more.  Not decided: minus infinity / infinity (also
// where squares may have come out below the smallest normal number, whose rounding is no fraction of them).
__device__ __forceinline__ float rough_least(const RoughRows& r, float sq, float norm) {
    const float d = (sqrtf(sq) * (1.f - kRoughTurn - r.slack) - 2 * r.turn * norm - r.tiny) * (1.f - kRoughTurn - r.slack);
    return sq < 1e37f && sq > 1e-30f ? d : -__builtin_inff();
}
__device__ __forceinline__ float rough_most(const RoughRows& r, float sq, float norm) {
    const float d = (sqrtf(sq) * (1.f + 1.01f * kRoughTurn + r.slack) + 2 * r.turn * norm + r.tiny) * (1.f + 1.01f * kRoughTurn + r.slack);
    return sq < 1e37f && sq > 1e-30f ? d : __builtin_inff();
}

// Sum over each group of LPR lanes; every lane of a group ends with the group's total.
template <int DIMV>
__device__ __forceinline__ float row_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false));  // row_half_mirror
    if constexpr (RowShape<DIMV>::LPR >= 16)
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, false));  // row_mirror
    if constexpr (RowShape<DIMV>::LPR >= 32) v += lane_xor<16>(v);
    if constexpr (RowShape<DIMV>::LPR >= 64) v += lane_xor<32>(v);
    return v;
}

// Squared distance of a row to a reference row, both spread over a group of lanes; every lane of a group ends with it.
template <int DIMV>
__device__ __forceinline__ float byte_sqdist(const RowRegs<DIMV>& ref, const uint4& x) {
    static_assert(RowShape<DIMV>::BYTES, "rows of bytes");
    int v = static_cast<int>(dot_bytes(x, x, ref.sq)) - 2 * static_cast<int>(dot_bytes(ref.v, x, 0u));
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false);   // row_half_mirror
    if constexpr (RowShape<DIMV>::LPR >= 16) v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false);   // row_mirror
    asm("" : "+v"(v));   // the last addition stays with its lane move (in the one lane that writes the sum it would be three instructions)
    return static_cast<float>(v);
}

// reference distance.cuh:22-26: Euclidean reports sqrt, Cosine the squared L2 of pre-normalised rows
__device__ __forceinline__ float finish_distance(float sq, int metric) { return metric == kEuclidean ? sqrtf(sq) : sq; }

// The same for a whole number below 2^24, the squared distance of rows of bytes: sqrtf without the scaling it needs for very
// small arguments and without the cases of infinity and NaN, half of its fourteen instructions.  The hardware root is off by
// one place at most; with neighbours l and h of it, l * root >= sq says that it is too large, h * root < sq that it is too small
// (both exact in the sign of one rounded multiply-add): Tuckerman's test, from Agarwal, Cooley, Gustavson, Shearer, Slishman and
// Tuckerman, "New scalar and vector elementary functions for the IBM System/370", IBM J. Res. Dev. 30 (1986) 126.
__device__ __forceinline__ float finish_byte_distance(float sq, int metric) {
    if (metric != kEuclidean) return sq;
    const float root = __builtin_amdgcn_sqrtf(sq);
    const float l = __uint_as_float(__float_as_uint(root) - 1u), h = __uint_as_float(__float_as_uint(root) + 1u);   // l of 0 is no number: neither test holds
    const float below = fmaf(-l, root, sq), above = fmaf(-h, root, sq);
    const float r = below <= 0.f ? l : root;
    return above > 0.f ? h : r;
}
template <int DIMV>
__device__ __forceinline__ float finish_row_distance(float sq, int metric) {
    if constexpr (RowShape<DIMV>::BYTES) return finish_byte_distance(sq, metric);
    else return finish_distance(sq, metric);
}

}  // namespace glide
