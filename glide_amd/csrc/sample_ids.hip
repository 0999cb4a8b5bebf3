// The rows of a k-means sample: the first `count` places of a seeded random permutation of 0 .. num-1.
// Reference: partition.cuh:30-44 (iota, std::shuffle with a random seed, the first sample_num entries).
//
// The permutation is a Fisher-Yates shuffle from the top -- for i = num-1 .. 1: swap places i and j_i, j_i uniform in 0 .. i --
// whose j_i are drawn from the PCG64 generator (O'Neill 2014: a 128-bit linear congruential generator, output xor-folded and
// rotated) by masked rejection: 32 bits at a time, the lower half of an output before the upper one, cut to the bits of i,
// drawn again while above i.  That is how numpy's Generator.permutation comes to its order, so a sample is the one that the
// host layer's seeds have always given.  On the host, shuffling two million ids to keep 20 000 of them took 13 ms, half of
// the whole partitioning; here it is
//   1. the generator's output, any part of which can be reached by jumping ahead (sample_stream_kernel),
//   2. which draw belongs to which i: a chain, since a draw is refused or taken by the i that the draws before it have left
//      (sample_accept_kernel, one workgroup),
//   3. the source of each place kept: place p holds what stood at j_p before step p and what step p found there is what the
//      steps before had moved: backwards in time, that is the place i of the next step i > p with j_i = j_p, then of the next
//      one with j = i, and so on.  Lists of the steps by their j answer that (sample_link_kernel, sample_trace_kernel).
#include "common.hpp"
#include "host_util.hpp"

namespace glide {

typedef unsigned __int128 u128;

constexpr uint32_t kDrawThreads = 1024, kDrawsPerThread = 16;
constexpr uint32_t kDrawChunk = kDrawThreads * kDrawsPerThread;   // draws settled at a time

struct Lcg {   // x -> a x + c
    u128 a, c;
};
__host__ __device__ inline Lcg lcg_then(const Lcg& first, const Lcg& second) { return Lcg{second.a * first.a, second.a * first.c + second.c}; }
__host__ __device__ inline Lcg lcg_steps(Lcg one, unsigned long long steps) {   // `one` applied `steps` times
    Lcg all{1, 0};
    for (; steps; steps >>= 1) {
        if (steps & 1) all = lcg_then(all, one);
        one = lcg_then(one, one);
    }
    return all;
}
__host__ inline Lcg pcg64_step(u128 increment) { return Lcg{(static_cast<u128>(0x2360ED051FC65DA4ull) << 64) | 0x4385DF649FCCF645ull, increment}; }
__device__ __forceinline__ unsigned long long pcg64_output(u128 state) {
    const unsigned long long hi = static_cast<unsigned long long>(state >> 64), folded = hi ^ static_cast<unsigned long long>(state);
    const uint32_t r = static_cast<uint32_t>(hi >> 58);
    return (folded >> r) | (folded << ((64 - r) & 63));
}

struct DrawArgs {
    u128 state;    // of the generator before its first output
    Lcg step;      // one output on
    Lcg thread;    // kDrawsPerThread / 2 outputs on
    Lcg block;     // 256 threads' worth on
};

// The kDrawsPerThread draws from number `first` (a multiple of it) on; `at` is the state before them.
__device__ __forceinline__ void make_draws(u128 at, const Lcg& step, uint32_t (&draw)[kDrawsPerThread]) {
#pragma unroll
    for (uint32_t k = 0; k < kDrawsPerThread; k += 2) {
        at = step.a * at + step.c;
        const unsigned long long o = pcg64_output(at);
        draw[k] = static_cast<uint32_t>(o);
        draw[k + 1] = static_cast<uint32_t>(o >> 32);
    }
}

// Draws in the order of the generator, sixteen a thread: bound by the 128-bit products (2.9M draws: 12 us).
__global__ __launch_bounds__(256) void sample_stream_kernel(DrawArgs a, uint32_t threads, uint32_t* stream) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= threads) return;
    const Lcg to_block = lcg_steps(a.block, blockIdx.x), to_thread = lcg_then(to_block, lcg_steps(a.thread, threadIdx.x));
    uint32_t draw[kDrawsPerThread];
    make_draws(to_thread.a * a.state + to_thread.c, a.step, draw);
    uint4* out = reinterpret_cast<uint4*>(stream + static_cast<size_t>(i) * kDrawsPerThread);
#pragma unroll
    for (uint32_t k = 0; k < kDrawsPerThread; k += 4) out[k / 4] = make_uint4(draw[k], draw[k + 1], draw[k + 2], draw[k + 3]);
}

// What a thread's draws settle: the i of the first one, and which of them are taken (the k-th taken one is the j of i - k).
struct Settled {
    uint32_t from, taken;   // a bit a draw
};
__device__ __forceinline__ uint32_t cut(uint32_t draw, uint32_t i) { return draw & (0xffffffffu >> __clz(static_cast<int>(i | 1u))); }   // to the bits of i

// heads[v] and links chain all i > v with j_i = v, in no particular order; steps[p] = j_p of the places kept.
__device__ __forceinline__ void link_steps(const uint32_t (&draw)[kDrawsPerThread], Settled s, uint32_t count, uint32_t* heads, uint32_t* links, uint32_t* steps) {
    uint32_t i = s.from;
#pragma unroll
    for (uint32_t k = 0; k < kDrawsPerThread; k++) {
        if ((s.taken >> k) & 1u) {
            const uint32_t v = cut(draw[k], i);
            if (v != i) links[i] = atomicExch(&heads[v], i);
            if (i < count) steps[i] = v;
            i--;
        }
    }
}
__device__ __forceinline__ void load_draws(const uint32_t* stream, size_t thread, uint32_t (&draw)[kDrawsPerThread]) {
    const uint4* in = reinterpret_cast<const uint4*>(stream + thread * kDrawsPerThread);
#pragma unroll
    for (uint32_t k = 0; k < kDrawsPerThread; k += 4) {
        const uint4 q = in[k / 4];
        draw[k] = q.x; draw[k + 1] = q.y; draw[k + 2] = q.z; draw[k + 3] = q.w;
    }
}

// Which draw belongs to which i, a chunk of 16 384 draws at a time.  A thread holds sixteen consecutive draws and walks them
// from the i it assumes the draws before have left; a scan over the taken counts corrects the assumption.  A correction by
// less than the distance between every draw and its i changes no draw's fate (no i of the chunk may have another number of
// bits for that, or the draws would be cut differently), so hardly any thread walks again; the rounds go on until nobody
// has, which a thread can cause at most once for every thread before it.  Two barriers a round, one round as a rule: the
// chain is what the whole draw waits for (2M ids: 0.4 of 0.5 ms).  Draws beyond `ready` chunks of the stream -- it holds two
// for every i and 1.4 are expected -- are made and linked on the spot.
__global__ __launch_bounds__(kDrawThreads) void sample_accept_kernel(DrawArgs a, uint32_t num, uint32_t count, const uint32_t* stream, uint32_t ready,
                                                                     Settled* settled, uint32_t* heads, uint32_t* links, uint32_t* steps) {
    __shared__ __attribute__((aligned(16))) uint32_t wave_total[2][kDrawThreads / 64];
    __shared__ uint32_t again[2];   // whether a thread has to walk once more, by the parity of the round
    const int lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t top = num - 1;   // the i of the chunk's first draw
    uint32_t parity = 0, chunk = 0;
    uint32_t draw[kDrawsPerThread], next[kDrawsPerThread];
    load_draws(stream, threadIdx.x, next);
    for (; top > 0; chunk++) {
#pragma unroll
        for (uint32_t k = 0; k < kDrawsPerThread; k++) draw[k] = next[k];
        if (chunk + 1 < ready) {
            load_draws(stream, static_cast<size_t>(chunk + 1) * kDrawThreads + threadIdx.x, next);
        } else {
            const Lcg to = lcg_steps(a.thread, static_cast<unsigned long long>(chunk + 1) * kDrawThreads + threadIdx.x);
            make_draws(to.a * a.state + to.c, a.step, next);
        }
        const uint32_t bits = 32 - __clz(static_cast<int>(top));
        const bool one_cut = top > kDrawChunk && 32 - __clz(static_cast<int>(top - kDrawChunk)) == static_cast<int>(bits);
        const float rate = static_cast<float>(top) / static_cast<float>(0xffffffffu >> (32 - bits));
        const uint32_t guess = static_cast<uint32_t>(rate * static_cast<float>(threadIdx.x * kDrawsPerThread));
        Settled s{top > guess ? top - guess : 0u, 0u};
        uint32_t total, slack = 0;
        bool walk = true;
        do {
            if (walk) {
                uint32_t i = s.from;
                s.taken = 0;
                slack = 0xffffffffu;
#pragma unroll
                for (uint32_t k = 0; k < kDrawsPerThread; k++) {
                    // i == 0: nothing is left to draw for
                    const uint32_t v = cut(draw[k], i);
                    const bool take = i != 0 && v <= i;
                    const uint32_t off = v <= i ? i - v : v - i - 1;   // how far i can move and the draw's fate not
                    slack = off < slack ? off : slack;
                    s.taken |= take ? 1u << k : 0u;
                    i -= take ? 1u : 0u;
                }
                if (!one_cut) slack = 0;
            }
            const uint32_t mine = __popc(s.taken);
            uint32_t in_wave;
            const uint32_t before_in_wave = wave_exclusive_scan(mine, in_wave);
            if (lane == 0) wave_total[parity][wave] = in_wave;
            if (threadIdx.x == 0) again[parity] = 0;
            __syncthreads();
            uint32_t before = 0;
            total = 0;
#pragma unroll
            for (uint32_t w = 0; w < kDrawThreads / 64; w++) {
                const uint32_t t = wave_total[parity][w];
                before += w < wave ? t : 0u;
                total += t;
            }
            const uint32_t taken_before = before + before_in_wave, now = top > taken_before ? top - taken_before : 0u;
            const uint32_t moved = now > s.from ? now - s.from : s.from - now;
            walk = moved > slack;
            slack -= moved < slack ? moved : slack;   // what is left of it for the next correction
            s.from = now;
            if (ballot(walk) != 0 && lane == 0) again[parity] = 1;
            __syncthreads();
            parity ^= 1;   // the next round writes the other words: nobody is still reading those
        } while (again[parity ^ 1] != 0);
        if (chunk < ready)
            settled[static_cast<size_t>(chunk) * kDrawThreads + threadIdx.x] = s;
        else
            link_steps(draw, s, count, heads, links, steps);
        top -= total < top ? total : top;
    }
    for (; chunk < ready; chunk++) settled[static_cast<size_t>(chunk) * kDrawThreads + threadIdx.x] = Settled{0u, 0u};
}

__global__ __launch_bounds__(256) void sample_link_kernel(uint32_t threads, uint32_t count, const uint32_t* stream, const Settled* settled, uint32_t* heads,
                                                          uint32_t* links, uint32_t* steps) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= threads) return;
    const Settled s = settled[t];
    if (s.taken == 0) return;
    uint32_t draw[kDrawsPerThread];
    load_draws(stream, t, draw);
    link_steps(draw, s, count, heads, links, steps);
}

__global__ __launch_bounds__(256) void sample_trace_kernel(uint32_t count, const uint32_t* steps, const uint32_t* heads, const uint32_t* links, uint32_t* ids) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= count) return;
    uint32_t place = p == 0 ? 0u : steps[p], time = p;
    for (;;) {
        uint32_t next = kInvalid;   // the first step after `time` that swaps with `place`
        for (uint32_t i = heads[place]; i != kInvalid; i = links[i])
            if (i > time && i < next) next = i;
        if (next == kInvalid) break;
        place = time = next;
    }
    ids[p] = place;
}

}  // namespace glide

using namespace glide;

extern "C" {

namespace {
constexpr uint32_t kMostIds = 1u << 30;   // threads of the stream are counted with 32 bits
struct SampleLayout { size_t stream, settled, heads, links, steps, total; uint32_t chunks; };
SampleLayout sample_layout(uint32_t num) {
    SampleLayout l;
    l.chunks = static_cast<uint32_t>((static_cast<size_t>(num) * 2 + kDrawChunk - 1) / kDrawChunk);   // two draws for every i, whole chunks
    size_t off = 0;
    auto take = [&off](size_t bytes) { const size_t o = off; off += (bytes + 15) / 16 * 16; return o; };
    l.stream = take(static_cast<size_t>(l.chunks) * kDrawChunk * 4);
    l.settled = take(static_cast<size_t>(l.chunks) * kDrawThreads * sizeof(Settled));
    l.heads = take(static_cast<size_t>(num) * 4);
    l.links = take(static_cast<size_t>(num) * 4);
    l.steps = take(static_cast<size_t>(num) * 4);
    l.total = off;
    return l;
}
}  // namespace

size_t glide_hip_sample_ids_workspace_bytes(uint32_t num) { return num <= kMostIds ? sample_layout(num).total : 0; }

int glide_hip_sample_ids(uint32_t num, uint32_t count, const uint64_t* generator, uint32_t* ids, void* workspace, size_t workspace_bytes, void* stream) {
    if (!generator || !ids || !workspace || num == 0 || count > num) return GLIDE_ERR_BAD_ARGUMENT;
    if (num > kMostIds) return GLIDE_ERR_UNSUPPORTED;
    const SampleLayout l = sample_layout(num);
    if (workspace_bytes < l.total || reinterpret_cast<uintptr_t>(workspace) % 16) return GLIDE_ERR_BAD_ARGUMENT;
    if (count == 0) return GLIDE_OK;
    hipStream_t s = as_stream(stream);
    unsigned char* w = static_cast<unsigned char*>(workspace);
    uint32_t* draws = reinterpret_cast<uint32_t*>(w + l.stream);
    Settled* settled = reinterpret_cast<Settled*>(w + l.settled);
    uint32_t* heads = reinterpret_cast<uint32_t*>(w + l.heads);
    uint32_t* links = reinterpret_cast<uint32_t*>(w + l.links);
    uint32_t* steps = reinterpret_cast<uint32_t*>(w + l.steps);
    DrawArgs a;
    a.state = (static_cast<u128>(generator[0]) << 64) | generator[1];
    a.step = pcg64_step((static_cast<u128>(generator[2]) << 64) | generator[3]);
    a.thread = lcg_steps(a.step, kDrawsPerThread / 2);
    a.block = lcg_steps(a.thread, 256);
    const uint32_t threads = l.chunks * kDrawThreads;
    const int rc = glide_hip_fill_u32(heads, kInvalid, num, stream);
    if (rc != GLIDE_OK) return rc;
    hipLaunchKernelGGL(sample_stream_kernel, dim3(threads / 256), dim3(256), 0, s, a, threads, draws);
    hipLaunchKernelGGL(sample_accept_kernel, dim3(1), dim3(kDrawThreads), 0, s, a, num, count, draws, l.chunks, settled, heads, links, steps);
    hipLaunchKernelGGL(sample_link_kernel, dim3(threads / 256), dim3(256), 0, s, threads, count, draws, settled, heads, links, steps);
    hipLaunchKernelGGL(sample_trace_kernel, dim3(ceil_div(count, 256)), dim3(256), 0, s, count, steps, heads, links, ids);
    return launch_status();
}

}  // extern "C"
