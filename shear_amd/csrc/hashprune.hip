// hashprune.hip -- HashPrune reservoirs on the GPU: the reducer that consumes
// the edge-record stream (SpillRecord16) and keeps, per source point, at most
// l_max neighbours.
//
// Reference semantics (shear-core/src/algorithm/pipnn/): HashPruneReservoir
// insert (hash_prune.rs:1333-1453) under the total order (dist by total_cmp,
// target, hash; :2094-2106), fed edge by edge by the spill reducer
// (spill_hashprune.rs:2686-2719) and emitted as the slot targets in slot
// order, ascending hash (:3203-3221 emit_shard).  With the backfill and
// evidence policies off (params.rs:3346-3350) that reservoir ends in a state
// that depends only on the set of candidates inserted: each hash keeps its
// best candidate (a hit keeps the better one), and of those the l_max best
// remain (an evicted or rejected candidate is worse than l_max others of
// distinct hashes, and those are only ever replaced by better ones).  So a
// batch of records can be merged in any order, which is what makes it a GPU
// reduction.  Record batches:
//   1. count records per source (atomics), exclusive scan, list the sources that
//      have any, scatter the records grouped by source (the per-source counters
//      return to zero);
//   2. one wave per listed source merges its slots with its records
//      (hp_merge_kernel).
// Segment batches (records left where the emitter wrote them, described by
// per-source runs) are merged in place by the same kernel.  Between merges
// the slots are kept in no particular order; the export sorts each reservoir
// by hash, the reference's emit order.
#include <hipcub/hipcub.hpp>

#include "hashprune_kernels.h"

namespace tessa {

namespace {

constexpr int kHpWaves = 4;                 // waves per workgroup of the merge kernels
constexpr uint32_t kHpMergeGrid = 4096;     // workgroups of a merge, each walking its share of the sources
constexpr int kHpThreads = kHpWaves * 64;
constexpr int kScanThreads = 1024;
constexpr int kScanPerThread = 4;
constexpr uint32_t kScanBlock = kScanThreads * kScanPerThread;

__device__ __forceinline__ uint32_t total_key(float d) {
    const uint32_t b = __float_as_uint(d);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_dist(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v, uint32_t lane, uint32_t &total) {
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= (uint32_t)off) x += y;
    }
    total = __shfl(x, 63);
    return x - v;
}

// Record batches: the sources that have records, each one's first grouped
// record and how many.  Sources of up to `few` records (0: none) are listed from
// the end of the arrays backwards, the others from the front; count: how many
// of each, [0] the others, [1] these.
__host__ __device__ inline uint32_t hp_few_records(uint32_t l_max) { return l_max <= 64u ? 20u : 32u; }
struct HpRuns {
    uint32_t *src, *start, *len, *count;
    uint32_t capacity, few;
};
HpRuns record_runs(const HashPruneState &s) {
    uint32_t *r = s.runs;
    return HpRuns{r,
                  r + s.runs_capacity,
                  r + 2 * s.runs_capacity,
                  reinterpret_cast<uint32_t *>(s.status + 1),
                  (uint32_t)s.runs_capacity,
                  s.rhalf_mode != 0 ? hp_few_records(s.l_max) : 0u};
}

__global__ void hp_fill_u32(uint32_t *a, uint64_t n, uint32_t v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = v;
}

// status[0]: first record with a bad source; status[1]: the lengths of a record batch's two lists.
__global__ void hp_status_init(uint64_t *status) {
    status[0] = ~0ull;
    status[1] = 0ull;
}

// Lanes of a wave holding the same source as the wave's first active lane
// share one atomic (the edge stream interleaves one row's outgoing records
// with its reverse ones, so about half a wave has the same source).
__device__ __forceinline__ uint64_t same_as_leader(uint32_t src, bool active, uint32_t &leader_src) {
    const uint64_t act = __ballot(active);
    const uint32_t leader = act ? (uint32_t)__builtin_ctzll(act) : 0u;
    leader_src = __shfl(src, leader);
    return __ballot(active && src == leader_src);
}

__global__ void hp_count_kernel(const uint4 *rec, uint64_t count, uint32_t num_points, uint32_t *bucket,
                                uint64_t *status) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    // uniform trip count per wave: lanes past the end stay inactive
    for (uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u); i0 < count; i0 += stride) {
        const uint64_t i = i0 + lane;
        const bool in = i < count;
        const uint32_t src = in ? rec[i].x : 0u;
        const bool bad = in && src >= num_points;
        if (bad) atomicMin((unsigned long long *)status, (unsigned long long)i);
        uint32_t lsrc;
        const uint64_t grp = same_as_leader(src, in && !bad, lsrc);
        const bool in_grp = (grp >> lane) & 1ull;
        if (in_grp && lane == (uint32_t)__builtin_ctzll(grp)) atomicAdd(&bucket[lsrc], (uint32_t)__popcll(grp));
        if (in && !bad && !in_grp) atomicAdd(&bucket[src], 1u);
    }
}

// Block sums of `bucket` over kScanBlock elements each.
__global__ __launch_bounds__(kScanThreads) void hp_scan_reduce(const uint32_t *bucket, uint32_t n, uint32_t *sums) {
    __shared__ uint32_t ws[kScanThreads / 64];
    const uint32_t base = blockIdx.x * kScanBlock + threadIdx.x * kScanPerThread;
    uint32_t v = 0;
#pragma unroll
    for (int e = 0; e < kScanPerThread; ++e) v += base + e < n ? bucket[base + e] : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if ((threadIdx.x & 63u) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kScanThreads / 64; ++w) t += ws[w];
        sums[blockIdx.x] = t;
    }
}

// Exclusive scan of the block sums in place (one workgroup); offsets[n] = total.
__global__ __launch_bounds__(kScanThreads) void hp_scan_partials(uint32_t *sums, uint32_t nb, uint32_t *offsets,
                                                                 uint32_t n) {
    __shared__ uint32_t ws[kScanThreads / 64];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t b0 = 0; b0 < nb; b0 += kScanThreads) {
        const uint32_t i = b0 + threadIdx.x;
        const uint32_t v = i < nb ? sums[i] : 0u;
        uint32_t wt;
        const uint32_t ex = wave_excl_scan(v, lane, wt);
        if (lane == 0) ws[wave] = wt;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < kScanThreads / 64; ++w) {
            before += w < wave ? ws[w] : 0u;
            all += ws[w];
        }
        if (i < nb) sums[i] = carry + before + ex;
        __syncthreads();
        if (threadIdx.x == 0) carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) offsets[n] = carry;
}

// Every source's first grouped record, and the lists of the sources that have
// any: the merge takes these only (walking all points of a set of 10 M for 1,000
// records took 2.0 ms, all of the insert with the list 0.1).  Blocks append in
// any order.
__global__ __launch_bounds__(kScanThreads) void hp_scan_apply(const uint32_t *bucket, uint32_t n, const uint32_t *sums,
                                                              uint32_t *offsets, HpRuns runs) {
    __shared__ uint32_t ws[kScanThreads / 64], wa[kScanThreads / 64], at0[2];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t base = blockIdx.x * kScanBlock + threadIdx.x * kScanPerThread;
    // listed: sources of more than `few` records in the low half, the others in the high one
    static_assert(kScanBlock < 0x10000u, "a block's sources fit 16 bits");
    uint32_t v[kScanPerThread], t = 0, listed = 0;
    auto list_of = [&](uint32_t records) { return records == 0u ? 0u : records > runs.few ? 1u : 0x10000u; };
#pragma unroll
    for (int e = 0; e < kScanPerThread; ++e) {
        v[e] = base + e < n ? bucket[base + e] : 0u;
        t += v[e];
        listed += list_of(v[e]);
    }
    uint32_t wt, wl;
    const uint32_t ex = wave_excl_scan(t, lane, wt), el = wave_excl_scan(listed, lane, wl);
    if (lane == 0) {
        ws[wave] = wt;
        wa[wave] = wl;
    }
    __syncthreads();
    uint32_t before = sums[blockIdx.x], ahead = 0;
    for (uint32_t w = 0; w < wave; ++w) {
        before += ws[w];
        ahead += wa[w];
    }
    if (threadIdx.x == kScanThreads - 1u) {
        const uint32_t all = ahead + wl;
        at0[0] = (all & 0xffffu) ? atomicAdd(&runs.count[0], all & 0xffffu) : 0u;
        at0[1] = (all >> 16) ? atomicAdd(&runs.count[1], all >> 16) : 0u;
    }
    __syncthreads();
    uint32_t run = before + ex, many = at0[0] + ((ahead + el) & 0xffffu), few = at0[1] + ((ahead + el) >> 16);
#pragma unroll
    for (int e = 0; e < kScanPerThread; ++e) {
        if (base + e < n) offsets[base + e] = run;
        if (v[e] != 0u) {
            const uint32_t at = v[e] > runs.few ? many++ : runs.capacity - 1u - few++;
            runs.src[at] = base + e;
            runs.start[at] = run;
            runs.len[at] = v[e];
        }
        run += v[e];
    }
}

// Records grouped by source; the per-source counters count back down to zero.
__global__ void hp_scatter_kernel(const uint4 *rec, uint64_t count, uint32_t num_points, uint32_t *bucket,
                                  const uint32_t *offsets, uint4 *grouped) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u); i0 < count; i0 += stride) {
        const uint64_t i = i0 + lane;
        const bool in = i < count;
        const uint4 r = in ? rec[i] : make_uint4(0u, 0u, 0u, 0u);
        const bool ok = in && r.x < num_points;
        uint32_t lsrc;
        const uint64_t grp = same_as_leader(r.x, ok, lsrc);
        const bool in_grp = (grp >> lane) & 1ull;
        // the group takes popcount(grp) positions with one atomic; lane order inside it
        const uint32_t first = grp ? (uint32_t)__builtin_ctzll(grp) : 0u;
        uint32_t top = 0;
        if (in_grp && lane == first) top = atomicSub(&bucket[lsrc], (uint32_t)__popcll(grp));
        top = __shfl(top, first);
        if (in_grp) {
            const uint32_t below = (uint32_t)__popcll(grp & ((1ull << lane) - 1ull));
            grouped[offsets[lsrc] + top - 1u - below] = r;
        } else if (ok) {
            grouped[offsets[r.x] + atomicSub(&bucket[r.x], 1u) - 1u] = r;
        }
    }
}

template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xf, 0xf, false);
}
// The value of lane ^ j (j a power of two, known at compile time): data moves
// inside a row of 16 lanes cost no LDS operation.
template <uint32_t j>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (j == 1u) return dpp_mov<0xb1>(v);                 // quad_perm [1,0,3,2]
    else if constexpr (j == 2u) return dpp_mov<0x4e>(v);            // quad_perm [2,3,0,1]
    else if constexpr (j == 4u) return dpp_mov<0x141>(dpp_mov<0x1b>(v));  // half mirror (^7) of quad_perm [3,2,1,0] (^3)
    else if constexpr (j == 8u) return dpp_mov<0x128>(v);           // rotation of a row by 8
    else return __shfl_xor(v, (int)j);
}

// Ascending bitonic sort of 64 * E values, value q * 64 + lane in register q.
template <int E, uint32_t kk, uint32_t j>
__device__ __forceinline__ void sort_step(uint32_t (&x)[E], uint32_t lane) {
    if constexpr (j >= 64u) {
#pragma unroll
        for (int q = 0; q < E; ++q) {
            constexpr int jq = (int)(j / 64u);
            if ((q & jq) != 0) continue;
            const bool up = (((uint32_t)q * 64u) & kk) == 0u;  // kk > 64 here
            const uint32_t a = x[q], b = x[q | jq], lo = a < b ? a : b, hi = a < b ? b : a;
            x[q] = up ? lo : hi;
            x[q | jq] = up ? hi : lo;
        }
    } else {
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const uint32_t o = lane_xor<j>(x[q]);
            const bool up = (((uint32_t)q * 64u + lane) & kk) == 0u;
            const bool low = ((lane & j) == 0u) == up;
            const uint32_t lo = x[q] < o ? x[q] : o, hi = x[q] < o ? o : x[q];
            x[q] = low ? lo : hi;
        }
    }
    if constexpr (j > 1u) sort_step<E, kk, j / 2u>(x, lane);
}
template <int E, uint32_t kk = 2u>
__device__ __forceinline__ void sort_values(uint32_t (&x)[E], uint32_t lane) {
    sort_step<E, kk, kk / 2u>(x, lane);
    if constexpr (kk < 64u * E) sort_values<E, kk * 2u>(x, lane);
}

// A reservoir's slots in ascending hash order (the hashes are distinct): one
// word per slot, hash and position, is sorted, then the keys are fetched from
// their positions.  h: the hash, 0xffffffff for an unused slot (after the used
// ones); k: the key.
template <int E>
__device__ __forceinline__ void sort_slots(uint32_t (&h)[E], uint64_t (&k)[E], uint32_t lane) {
    uint32_t x[E];
#pragma unroll
    for (int q = 0; q < E; ++q) x[q] = h[q] > 0xffffu ? 0xffffffffu : (h[q] << 8) | ((uint32_t)q * 64u + lane);
    sort_values<E>(x, lane);
    uint64_t r[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const uint32_t from = x[q] & 63u, reg = (x[q] >> 6) & 3u;
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const uint32_t l = __shfl((uint32_t)k[p], (int)from), m = __shfl((uint32_t)(k[p] >> 32), (int)from);
            lo = reg == (uint32_t)p ? l : lo;
            hi = reg == (uint32_t)p ? m : hi;
        }
        r[q] = ((uint64_t)hi << 32) | lo;
        h[q] = x[q] == 0xffffffffu ? 0xffffffffu : x[q] >> 8;
    }
#pragma unroll
    for (int q = 0; q < E; ++q) k[q] = r[q];
}

// ---- segment mode: records left where the emitter put them ------------------
// A segment {src, first record lo/hi, count} names a run of records of one
// source.  The batch's segments are sorted by source (radix sort of the
// segment indices), each run of equal sources becomes one active source, and
// the merges walk the active sources only, reading each one's records in
// place: the work follows the batch size, with no pass over all points and
// no atomics per record.

__global__ void hp_seg_keys_kernel(const uint4 *segs, uint64_t nseg, uint32_t num_points, uint32_t *keys,
                                   uint32_t *vals, uint64_t *status) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nseg; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint4 g = segs[i];
        const bool bad = g.w != 0u && g.x >= num_points;
        // the first record of the segment carries the bad source
        if (bad) atomicMin((unsigned long long *)status, (unsigned long long)(((uint64_t)g.z << 32) | g.y));
        keys[i] = (g.w == 0u || bad) ? num_points : g.x;  // empty and bad segments sort last, unused
        vals[i] = (uint32_t)i;
    }
}

// The segment descriptors in sorted order (one gather, so the merge reads a
// source's segments contiguously).
__global__ void hp_seg_gather_kernel(const uint4 *segs, const uint32_t *order, uint64_t nseg, uint4 *sorted) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nseg; i += (uint64_t)gridDim.x * blockDim.x)
        sorted[i] = segs[order[i]];
}

// ---- merge ---------------------------------------------------------------------
// One wave per source with new records.  A batch of the source's records (64 *
// kHpNew of them, in registers beside its slots) is reduced at once instead of
// record by record:
//   1. a full reservoir drops the candidates past its worst distance;
//   2. each hash's best is found through a small table in LDS (best_of_hash):
//      every candidate takes the minimum of its bucket, the one that finds its
//      own key there claims the bucket and leaves its hash as a tag, and the
//      others see from the tag whether they lost to their own hash or only
//      share the bucket with another one (those try again);
//   3. when more than l_max hashes remain, the l_max best are the ones up to a
//      distance found by bisection, counting with ballots (keep_best); equal
//      distances at the border are settled by target, then hash;
//   4. the survivors are packed through LDS into the slots.
// What bounds it is latency (the memory pipeline below, then the dependent LDS
// steps at four waves per SIMD): about 300 vector and 470 scalar instructions
// and 40 LDS operations for a source with 128 records.  Inserting the
// candidates one by one (a rank ballot, a hash ballot and a shift each) took
// 88 SIMD cycles a record: 67 M records of 524,288 points 2.45 ms, by batches
// 0.73 ms.  Larger tables (fewer candidates try again) or five waves per SIMD
// (registers spill: 0.89 ms) cost more.  With the groups of a backfill policy
// the merges of a 1 M x 768 build take 3.5 ms in all.
constexpr int kHpNew = 4;              // new records per lane in one batch
constexpr uint32_t kHpBuckets = 1024;  // per wave; >= kHpMaxLMax (staging of the slots), a power of two

struct HpWaveLds {
    uint64_t key[kHpBuckets];  // ~0 between uses
};

__device__ __forceinline__ uint64_t readlane64(uint64_t v, uint32_t l) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)l) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)l);
}
__device__ __forceinline__ uint32_t readlane32(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ uint64_t ballot64(bool pred) { return __builtin_amdgcn_ballot_w64(pred); }
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }
__device__ __forceinline__ uint32_t below(uint64_t mask) {  // set bits of mask under this lane
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
// The lanes of positions [q * 64, q * 64 + 64) below n.
__device__ __forceinline__ uint64_t lanes_below(uint32_t n, uint32_t q) {
    const uint32_t m = n > q * 64u ? n - q * 64u : 0u;
    return m >= 64u ? ~0ull : (1ull << m) - 1ull;
}

// The wave's LDS operations complete in order; this keeps the compiler to it.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, true);
}
// Largest value of the wave (row shifts by 1, 2, 4, 8, then the row ends carried over).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    uint32_t o;
    o = dpp_or_zero<0x111>(v), v = v > o ? v : o;
    o = dpp_or_zero<0x112>(v), v = v > o ? v : o;
    o = dpp_or_zero<0x114>(v), v = v > o ? v : o;
    o = dpp_or_zero<0x118>(v), v = v > o ? v : o;
    o = dpp_or_zero<0x142>(v), v = v > o ? v : o;
    o = dpp_or_zero<0x143>(v), v = v > o ? v : o;
    return readlane32(v, 63u);
}

// Sets of candidates are lane masks, one per register (scalar registers, and a
// register without a candidate of the set costs one scalar branch).
//
// Among the candidates `in` (no key of ~0), win = the best key of each hash
// (one of several equal ones) and, when asked, rest = those of a winner's hash
// with another target than the winner's.
template <int R, bool kRest>
__device__ __forceinline__ void best_of_hash(HpWaveLds &t, const uint64_t (&k)[R], const uint32_t (&h)[R],
                                             const uint64_t (&in)[R], uint64_t (&win)[R], uint64_t (&rest)[R],
                                             uint32_t lane) {
    uint64_t pend[R], any = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        pend[q] = in[q];
        win[q] = 0;
        if (kRest) rest[q] = 0;
        any |= pend[q];
    }
    while (any) {
        uint64_t best[R], mark[R];
        // the bucket's best key
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (pend[q] && lane_in(pend[q]))
                __hip_atomic_fetch_min(&t.key[h[q] & (kHpBuckets - 1u)], k[q], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
        wave_lds_order();
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (pend[q]) best[q] = t.key[h[q] & (kHpBuckets - 1u)];
        wave_lds_order();
        // its owner (the last to write, when keys are equal) leaves its hash and position
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (pend[q] && lane_in(pend[q] & ballot64(best[q] == k[q])))
                t.key[h[q] & (kHpBuckets - 1u)] = ((uint64_t)h[q] << 32) | ((uint32_t)q * 64u + lane);
        wave_lds_order();
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (pend[q]) mark[q] = t.key[h[q] & (kHpBuckets - 1u)];
        wave_lds_order();
        any = 0;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (!pend[q]) continue;
            const uint64_t own = pend[q] & ballot64((uint32_t)mark[q] == (uint32_t)q * 64u + lane);
            const uint64_t same = pend[q] & ballot64((uint32_t)(mark[q] >> 32) == h[q]);
            if (lane_in(own)) t.key[h[q] & (kHpBuckets - 1u)] = ~0ull;
            win[q] |= own;
            if (kRest) rest[q] |= same & ~own & ballot64((uint32_t)best[q] != (uint32_t)k[q]);
            pend[q] &= ~same;
            any |= pend[q];
        }
        wave_lds_order();
    }
}

// Over the values v of the set m (more than `need` of them): a t with
// count(v <= t) == need if there is one, else the smallest t with more; cle =
// count(v <= t).  Each other step interpolates between the counts at the
// ends (the distances of a reservoir's candidates spread evenly enough for
// about 4 steps where bisection alone takes 10), the ones between halve.
template <int R>
__device__ __forceinline__ uint32_t kth_value(const uint32_t (&v)[R], const uint64_t (&m)[R], uint32_t need,
                                              uint32_t &cle) {
    uint32_t mx = 0, mn = 0, n = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const uint32_t a = lane_in(m[q]) ? v[q] : 0u, b = lane_in(m[q]) ? ~v[q] : 0u;
        mx = mx > a ? mx : a;
        mn = mn > b ? mn : b;
        n += (uint32_t)__popcll(m[q]);
    }
    // count(v <= hi) = c_hi >= need, count(v < lo) = c_lo < need
    uint32_t hi = wave_max_u32(mx), lo = ~wave_max_u32(mn), c_hi = n, c_lo = 0;
    bool halve = false;
    while (lo < hi) {
        const uint32_t span = hi - lo;
        uint32_t step = span / 2u;
        if (!halve) {
            const float f = (float)(need - c_lo) * __builtin_amdgcn_rcpf((float)(c_hi - c_lo));
            const uint32_t s = (uint32_t)(f * (float)span);
            step = (uint32_t)__builtin_amdgcn_readfirstlane((int)(s < span ? s : span - 1u));
        }
        halve = !halve;
        const uint32_t mid = lo + step;
        uint32_t c = 0;
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (m[q]) c += (uint32_t)__popcll(ballot64(v[q] <= mid) & m[q]);
        if (c == need) {
            cle = c;
            return mid;
        }
        if (c > need) {
            hi = mid;
            c_hi = c;
        } else {
            lo = mid + 1u;
            c_lo = c;
        }
    }
    cle = c_hi;
    return lo;
}

// Leaves the l_max best of the candidates win (more than l_max of them,
// distinct hashes) by (distance key, target, hash).
template <int R>
__device__ __forceinline__ void keep_best(const uint64_t (&k)[R], const uint32_t (&h)[R], uint64_t (&win)[R],
                                          uint32_t l_max) {
    uint32_t d[R], cle;
#pragma unroll
    for (int q = 0; q < R; ++q) d[q] = (uint32_t)(k[q] >> 32);
    const uint32_t td = kth_value<R>(d, win, l_max, cle);
    if (cle == l_max) {
#pragma unroll
        for (int q = 0; q < R; ++q) win[q] &= ballot64(d[q] <= td);
        return;
    }
    // candidates of the distance at the border: by target, then by hash
    uint64_t sure[R], eq[R];
    uint32_t need = l_max, tg[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
        sure[q] = win[q] & ballot64(d[q] < td);
        eq[q] = win[q] & ballot64(d[q] == td);
        tg[q] = (uint32_t)k[q];
        need -= (uint32_t)__popcll(sure[q]);
    }
    const uint32_t tt = kth_value<R>(tg, eq, need, cle);
    if (cle == need) {
#pragma unroll
        for (int q = 0; q < R; ++q) win[q] = sure[q] | (eq[q] & ballot64(tg[q] <= tt));
        return;
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const uint64_t lt = eq[q] & ballot64(tg[q] < tt);
        sure[q] |= lt;
        eq[q] &= ballot64(tg[q] == tt);
        need -= (uint32_t)__popcll(lt);
    }
    const uint32_t th = kth_value<R>(h, eq, need, cle);  // distinct hashes: exact
#pragma unroll
    for (int q = 0; q < R; ++q) win[q] = sure[q] | (eq[q] & ballot64(h[q] <= th));
}

// A wave's sources in the stages of its pipeline: the run (source, its sorted
// segments or its records [start, start + len); num_points: nothing to merge), the segments
// (lane s: segment s, cnt records from first), then the slots and the first
// batch of records (the lane's record q * 64 + lane of it, q < kHpNew).  Every
// load is unconditional, from a clamped address: a branch around a load
// costs a wait for it at the branch's end.
struct HpRun {
    uint32_t src, start, len;
};
struct HpSegs {
    uint32_t ng, cnt;
    uint64_t first;
};
template <int ER>
struct HpSlots {
    uint64_t k[ER];
    uint32_t h[ER], c;
};
struct HpBatch {
    uint32_t dst[kHpNew], hash[kHpNew], dist[kHpNew], total;  // hash: with the record's flags above 16 bits
};

struct HpMergeArgs {
    const uint4 *records;   // record batches: grouped by source
    const uint4 *sorted;    // segments by source
    // a source's records (record batches) or its sorted segments: [start, start + len)
    const uint32_t *run_src, *run_start, *run_len, *num_runs;
    uint32_t num_points, l_max, quota;
    uint64_t *slot_keys;
    uint16_t *slot_hash;
    uint32_t *slot_count;
    uint64_t *grp_keys;
};

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Run a of na; raw loads, made a run by hp_run_ready once they have arrived.
__device__ __forceinline__ HpRun hp_run_load(const HpMergeArgs &A, uint32_t a, uint32_t na) {
    const uint32_t i = a < na ? a : na - 1u;
    return HpRun{A.run_src[i], A.run_start[i], A.run_len[i]};
}
__device__ __forceinline__ HpRun hp_run_ready(const HpMergeArgs &A, const HpRun &l, uint32_t a, uint32_t na) {
    HpRun r{uniform(l.src), uniform(l.start), uniform(l.len)};
    const bool none = a >= na || r.src >= A.num_points;  // past the end, the run of empty / bad segments
    if (none) r = HpRun{A.num_points, 0u, 0u};
    return r;
}

// Segments [g0, g0 + 64) of a run; the same two steps.
template <bool kGrouped>
__device__ __forceinline__ uint4 hp_segs_load(const HpMergeArgs &A, const HpRun &r, uint32_t g0, uint32_t lane) {
    if (kGrouped) return make_uint4(r.src, r.start, 0u, r.len);
    const uint32_t s = g0 + lane;
    return A.sorted[(uint64_t)r.start + (s < r.len ? s : 0u)];
}
template <bool kGrouped>
__device__ __forceinline__ HpSegs hp_segs_ready(const HpRun &r, const uint4 &g, uint32_t g0, uint32_t lane) {
    const uint32_t left = kGrouped ? (r.len ? 1u : 0u) : r.len - g0;
    HpSegs s;
    s.ng = left < 64u ? left : 64u;
    s.cnt = lane < s.ng ? g.w : 0u;
    s.first = ((uint64_t)g.z << 32) | g.y;
    return s;
}

template <int ER>
__device__ __forceinline__ HpSlots<ER> hp_slots(const HpMergeArgs &A, uint32_t src, uint32_t lane) {
    HpSlots<ER> s;
    const uint32_t p = src < A.num_points ? src : 0u;
    const uint64_t base = (uint64_t)p * A.l_max;
    s.c = A.slot_count[p];
#pragma unroll
    for (int q = 0; q < ER; ++q) {
        // every slot position is read, not only the live ones: these loads do
        // not wait for the count
        const uint32_t e = (uint32_t)q * 64u + lane;
        s.k[q] = A.slot_keys[base + (e < A.l_max ? e : 0u)];
        s.h[q] = A.slot_hash[base + (e < A.l_max ? e : 0u)];
    }
    return s;
}

// Records [c0, c0 + 64 * kHpNew) of a group of segments, across their
// boundaries; lanes past the group's records read `safe`.
__device__ __forceinline__ void hp_batch(HpBatch &b, const uint4 *records, const uint4 *safe, const HpSegs &g,
                                         uint32_t c0, uint32_t lane) {
    uint32_t ps = 0;
    uint64_t at[kHpNew] = {};
    for (uint32_t s = 0; s < g.ng; ++s) {
        const uint64_t d = readlane64(g.first, s) - ps;
#pragma unroll
        for (int q = 0; q < kHpNew; ++q) at[q] = c0 + (uint32_t)q * 64u + lane >= ps ? d : at[q];
        ps += readlane32(g.cnt, s);
    }
    b.total = ps;
#pragma unroll
    for (int q = 0; q < kHpNew; ++q) {
        const uint32_t p = c0 + (uint32_t)q * 64u + lane;
        const uint4 *r = p < ps ? records + (at[q] + p) : safe;
        b.dst[q] = r->y;
        b.hash[q] = r->z;
        b.dist[q] = r->w;
    }
}

// Merges one batch of records into the reservoir (slots rk / rh at positions
// [0, c), in no particular order; with kRhalf and a free slot, each slot's
// group g).
template <int ER, bool kRhalf>
__device__ __forceinline__ void hp_absorb(HpWaveLds &t, const HpBatch &b, uint32_t c0, uint64_t (&rk)[ER],
                                          uint32_t (&rh)[ER], uint32_t &c, uint64_t (&g)[ER][kRhalfGroup],
                                          uint32_t l_max, uint32_t quota, uint32_t lane) {
    constexpr int S = ER + kHpNew;                               // slots, then new records
    constexpr int R = S + (kRhalf ? ER * (int)kRhalfGroup : 0);  // then group keys
    uint64_t k[R], in[R], win[R], rest[R];
    uint32_t h[R];
    uint32_t worst = 0xffffffffu;
    if (c == l_max) {
        uint32_t m = 0;
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const uint32_t d = lane_in(lanes_below(c, q)) ? (uint32_t)(rk[q] >> 32) : 0u;
            m = m > d ? m : d;
        }
        worst = wave_max_u32(m);
    }
    uint64_t fresh = 0, odd = 0;
#pragma unroll
    for (int q = 0; q < kHpNew; ++q) {
        const uint32_t dk = total_key(__uint_as_float(b.dist[q]));
        k[ER + q] = ((uint64_t)dk << 32) | b.dst[q];
        h[ER + q] = b.hash[q] & 0xffffu;
        in[ER + q] = lanes_below(b.total - c0, q) & ballot64(dk <= worst);
        fresh |= in[ER + q];
    }
    if (!fresh) return;
#pragma unroll
    for (int q = 0; q < ER; ++q) {
        k[q] = rk[q];
        h[q] = rh[q];
        in[q] = lanes_below(c, q);
    }
    // a key of ~0 (a NaN of all ones) takes no part in the buckets
#pragma unroll
    for (int q = 0; q < S; ++q) {
        const uint64_t o = in[q] & ballot64(k[q] == ~0ull);
        odd |= o;
        in[q] &= ~o;
    }
    if constexpr (kRhalf) {
#pragma unroll
        for (int q = 0; q < ER; ++q)
#pragma unroll
            for (uint32_t j = 0; j < kRhalfGroup; ++j) {
                const int i = S + q * (int)kRhalfGroup + (int)j;
                k[i] = g[q][j];
                h[i] = rh[q];
                in[i] = c < l_max ? lanes_below(c, q) & ballot64(g[q][j] != ~0ull) : 0ull;
            }
    }
    best_of_hash<R, kRhalf>(t, k, h, in, win, rest, lane);
    if (odd) {
        // it is the worst of any hash: kept if nothing else of its hash is
#pragma unroll
        for (int q = 0; q < S; ++q) {
            uint64_t m = ballot64(k[q] == ~0ull) &
                         (q < ER ? lanes_below(c, q) : lanes_below(b.total - c0, q - ER));
            while (m) {
                const uint32_t j = (uint32_t)__builtin_ctzll(m);
                const uint64_t bit = m & (0ull - m);
                m ^= bit;
                const uint32_t bh = readlane32(h[q], j);
                uint64_t held = 0;
#pragma unroll
                for (int p = 0; p < S; ++p) held |= win[p] & ballot64(h[p] == bh);
                if (!held) win[q] |= bit;
            }
        }
    }
    uint32_t n = 0;
#pragma unroll
    for (int q = 0; q < S; ++q) n += (uint32_t)__popcll(win[q]);
    if (n > l_max) {
        uint64_t ks[S], ws[S];
        uint32_t hs[S];
#pragma unroll
        for (int q = 0; q < S; ++q) ks[q] = k[q], hs[q] = h[q], ws[q] = win[q];
        keep_best<S>(ks, hs, ws, l_max);
#pragma unroll
        for (int q = 0; q < S; ++q) win[q] = ws[q];
        n = l_max;
    }
    // the survivors packed into the slots: keys, then hashes, through LDS
    uint32_t at = 0, pos[S];
#pragma unroll
    for (int q = 0; q < S; ++q) {
        pos[q] = at + below(win[q]);
        if (win[q] && lane_in(win[q])) t.key[pos[q]] = k[q];
        at += (uint32_t)__popcll(win[q]);
    }
    c = n;
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < ER; ++q) rk[q] = t.key[(uint32_t)q * 64u + lane];
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < S; ++q)
        if (win[q] && lane_in(win[q])) t.key[pos[q]] = h[q];
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < ER; ++q) {
        const bool live = lane_in(lanes_below(c, q));
        rh[q] = live ? (uint32_t)t.key[(uint32_t)q * 64u + lane] : 0xffffffffu;
        rk[q] = live ? rk[q] : ~0ull;
    }
    wave_lds_order();
#pragma unroll
    for (int q = 0; q < ER; ++q) t.key[(uint32_t)q * 64u + lane] = ~0ull;
    wave_lds_order();
    if constexpr (kRhalf) {
        if (c == l_max) return;  // a full reservoir stays full: its groups are never read again
        // the next best target of each hash, layer by layer
#pragma unroll
        for (int q = 0; q < ER; ++q)
#pragma unroll
            for (uint32_t j = 0; j < kRhalfGroup; ++j) g[q][j] = ~0ull;
        for (uint32_t layer = 0; layer < quota; ++layer) {
            uint64_t any = 0;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                in[q] = rest[q];
                any |= in[q];
            }
            if (!any) break;
            best_of_hash<R, true>(t, k, h, in, win, rest, lane);
#pragma unroll
            for (int q = 0; q < R; ++q) {
                uint64_t m = win[q];
                while (m) {
                    const uint32_t j = (uint32_t)__builtin_ctzll(m);
                    m &= m - 1ull;
                    const uint64_t bk = readlane64(k[q], j);
                    const uint32_t bh = readlane32(h[q], j);
#pragma unroll
                    for (int p = 0; p < ER; ++p)
#pragma unroll
                        for (uint32_t i = 0; i < kRhalfGroup; ++i)
                            g[p][i] = i == layer && rh[p] == bh ? bk : g[p][i];
                }
            }
        }
    }
}

// All vector loads in flight have arrived.
__device__ __forceinline__ void wait_loads() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0) only
    __builtin_amdgcn_sched_barrier(0);
}

// Each wave walks its sources (segment runs, or with kGrouped the sources of a
// record batch) with the next source's first batch and
// slots, and the one after's run, already in flight.  They are waited for
// after the merge and before its stores: a wait at their first use, in the
// next iteration, would also wait for the stores, and for the loads issued
// there (the branches between leave the compiler no exact count).
// Registers for four waves per SIMD up to 64 slots with groups: 133 left room for
// three (1,024 leaves of 1,024 rows, k 2, hashes of 4 to 12 bits: merge with its
// segments' sort 0.84-1.04 ms, then 0.79-0.93).
template <int ER, bool kRhalf, bool kGrouped>
__global__ __launch_bounds__(kHpThreads) __attribute__((amdgpu_waves_per_eu(ER == 1 && kRhalf ? 4 : 0))) void hp_merge_kernel(
    HpMergeArgs A) {
    __shared__ HpWaveLds lds[kHpWaves];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    HpWaveLds &t = lds[wave];
    const uint32_t waves = gridDim.x * kHpWaves;
    const uint32_t na = *A.num_runs;
    uint32_t a = blockIdx.x * kHpWaves + wave;
    if (a >= na) return;
    for (uint32_t i = lane; i < kHpBuckets; i += 64u) t.key[i] = ~0ull;
    wave_lds_order();
    const uint4 *safe = kGrouped ? A.records : A.sorted;
    // stages: slots and batch of source a, segments of the next, run of the one after
    HpRun raw = hp_run_load(A, a, na), raw1 = hp_run_load(A, a + waves, na),
          raw2 = hp_run_load(A, a + 2u * waves, na);
    HpRun run = hp_run_ready(A, raw, a, na), run1 = hp_run_ready(A, raw1, a + waves, na);
    uint4 seg = hp_segs_load<kGrouped>(A, run, 0u, lane), seg1 = hp_segs_load<kGrouped>(A, run1, 0u, lane);
    HpSegs segs = hp_segs_ready<kGrouped>(run, seg, 0u, lane);
    HpSlots<ER> slots = hp_slots<ER>(A, run.src, lane);
    HpBatch batch;
    hp_batch(batch, A.records, safe, segs, 0u, lane);
    wait_loads();
    for (; a < na; a += waves) {
        HpSegs segs1 = hp_segs_ready<kGrouped>(run1, seg1, 0u, lane);
        const HpRun run2 = hp_run_ready(A, raw2, a + 2u * waves, na);
        const HpSlots<ER> slots1 = hp_slots<ER>(A, run1.src, lane);
        HpBatch batch1;
        hp_batch(batch1, A.records, safe, segs1, 0u, lane);
        seg1 = hp_segs_load<kGrouped>(A, run2, 0u, lane);
        raw2 = hp_run_load(A, a + 3u * waves, na);
        uint64_t base = 0, rk[ER], g[ER][kRhalfGroup];
        uint32_t rh[ER], c = 0;
        if (run.src < A.num_points) {
            c = uniform(slots.c);
            base = (uint64_t)run.src * A.l_max;
#pragma unroll
            for (int q = 0; q < ER; ++q) {
                const uint32_t e = (uint32_t)q * 64u + lane;
                rk[q] = e < c ? slots.k[q] : ~0ull;
                rh[q] = e < c ? slots.h[q] : 0xffffffffu;
                if constexpr (kRhalf) {
#pragma unroll
                    for (uint32_t j = 0; j < kRhalfGroup; ++j)
                        g[q][j] = c < A.l_max && e < c ? A.grp_keys[(base + e) * kRhalfGroup + j] : ~0ull;
                }
            }
            for (uint32_t g0 = 0;;) {
                for (uint32_t c0 = 0;; c0 += 64u * kHpNew) {
                    if (g0 != 0u || c0 != 0u) hp_batch(batch, A.records, safe, segs, c0, lane);
                    hp_absorb<ER, kRhalf>(t, batch, c0, rk, rh, c, g, A.l_max, A.quota, lane);
                    if (batch.total - c0 <= 64u * kHpNew) break;
                }
                // a source with more than 64 segments in the batch: 64 at a time
                g0 += 64u;
                if (kGrouped || g0 >= run.len) break;
                segs = hp_segs_ready<false>(run, hp_segs_load<false>(A, run, g0, lane), g0, lane);
            }
        }
        wait_loads();
        if (run.src < A.num_points) {
#pragma unroll
            for (int q = 0; q < ER; ++q) {
                const uint32_t e = (uint32_t)q * 64u + lane;
                if (e < c) {
                    A.slot_keys[base + e] = rk[q];
                    A.slot_hash[base + e] = (uint16_t)rh[q];
                    if constexpr (kRhalf) {
                        if (c < A.l_max) {
#pragma unroll
                            for (uint32_t j = 0; j < kRhalfGroup; ++j)
                                A.grp_keys[(base + e) * kRhalfGroup + j] = g[q][j];
                        }
                    }
                }
            }
            if (lane == 0) A.slot_count[run.src] = c;
        }
        run = run1;
        run1 = run2;
        segs = segs1;
        slots = slots1;
        batch = batch1;
    }
}

// ---- few records of a source, with groups ------------------------------------
// A record batch's sources of up to hp_few_records records while a backfill
// policy keeps groups: the records go in one by one, each a hash ballot and an
// update of one lane's slot and group (a hash's best quota + 1 distinct targets
// in order), or an append, or in a full reservoir a replacement of its worst
// slot; only the lanes that changed are written back.  Merging a batch
// (hp_absorb) finds the groups anew, layer by layer, some 4,000 cycles however
// few the records.  1,000,000 sources, reservoirs of up to 30 slots, one by one
// and merged: one record each 446 and 1,138 us, 16 records 1.38 and 1.63 ms, 20
// 1.66 and 1.76, 24 2.02 and 1.93 (hashes drawn from 4,096); 20 records 1.67 and
// 2.97 ms, 32 2.61 and 3.47 (from 40).  More slots make a merge dearer: with 128,
// 32 records 3.60 and 3.65 ms (from 4,096), 3.63 and 6.68 (from 40).
struct HpFew {
    uint32_t src, start, len;
};
template <int ER>
struct HpFewData {
    uint64_t k[ER], g[ER][kRhalfGroup];
    uint32_t h[ER], c;
    uint4 rec;
};

// The run's slots, groups (of a reservoir with a free slot) and records.
template <int ER>
__device__ __forceinline__ void hp_few_load(HpFewData<ER> &d, const HpMergeArgs &A, const HpFew &r, uint32_t c,
                                            uint32_t lane) {
    const uint64_t base = (uint64_t)r.src * A.l_max;
    d.c = c;
    d.rec = A.records[r.start + (lane < r.len ? lane : 0u)];
#pragma unroll
    for (int q = 0; q < ER; ++q) {
        const uint32_t e = (uint32_t)q * 64u + lane, at = e < c ? e : 0u;
        d.k[q] = A.slot_keys[base + at];
        d.h[q] = A.slot_hash[base + at];
        const uint32_t ga = c < A.l_max ? at : 0u;
#pragma unroll
        for (uint32_t j = 0; j < kRhalfGroup; ++j) d.g[q][j] = A.grp_keys[(base + ga) * kRhalfGroup + j];
    }
}

template <int ER>
__global__ __launch_bounds__(kHpThreads) void hp_few_kernel(HpMergeArgs A, uint32_t capacity) {
    static_assert(kRhalfGroup == 3, "a slot and three group keys");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * kHpWaves;
    const uint32_t na = A.num_runs[1];
    uint32_t a = blockIdx.x * kHpWaves + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (a >= na) return;
    // raw loads; past the end the last run's, used by nobody
    auto run = [&](uint32_t i) {
        const uint32_t at = capacity - 1u - (i < na ? i : na - 1u);
        return HpFew{A.run_src[at], A.run_start[at], A.run_len[at]};
    };
    auto ready = [&](const HpFew &r) { return HpFew{uniform(r.src), uniform(r.start), uniform(r.len)}; };
    // stages: data of run a, count of the next, run of the one after
    HpFew raw2 = run(a + 2u * waves);
    HpFew r0 = ready(run(a)), r1 = ready(run(a + waves));
    HpFewData<ER> d0;
    hp_few_load<ER>(d0, A, r0, uniform(A.slot_count[r0.src]), lane);
    uint32_t c1 = A.slot_count[r1.src];
    wait_loads();
    for (; a < na; a += waves) {
        HpFewData<ER> d1;
        hp_few_load<ER>(d1, A, r1, uniform(c1), lane);
        const HpFew r2 = ready(raw2);
        c1 = A.slot_count[r2.src];
        raw2 = run(a + 3u * waves);
        const uint64_t base = (uint64_t)r0.src * A.l_max;
        const uint64_t key = ((uint64_t)total_key(__uint_as_float(d0.rec.w)) << 32) | d0.rec.y;
        const uint32_t hash = d0.rec.z & 0xffffu;
        uint64_t rk[ER], g[ER][kRhalfGroup], dirty[ER];
        uint32_t rh[ER], c = d0.c;
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const bool live = (uint32_t)q * 64u + lane < c;
            rk[q] = live ? d0.k[q] : ~0ull;
            rh[q] = live ? d0.h[q] : 0xffffffffu;
            dirty[q] = 0;
#pragma unroll
            for (uint32_t j = 0; j < kRhalfGroup; ++j) g[q][j] = live && c < A.l_max ? d0.g[q][j] : ~0ull;
        }
        for (uint32_t j = 0; j < r0.len; ++j) {
            const uint64_t k = readlane64(key, j);
            const uint32_t h = readlane32(hash, j);
            uint64_t hit[ER], any = 0;
#pragma unroll
            for (int q = 0; q < ER; ++q) {
                hit[q] = ballot64(rh[q] == h);
                any |= hit[q];
            }
            if (!any) {
                uint32_t place = c;
                if (c == A.l_max) {
                    // the worst slot by (distance, target, hash), if the record is better
                    uint64_t m[ER];
                    uint32_t worst[3];
#pragma unroll
                    for (int q = 0; q < ER; ++q) m[q] = lanes_below(c, q);
#pragma unroll
                    for (int w = 0; w < 3; ++w) {
                        uint32_t v[ER], top = 0;
#pragma unroll
                        for (int q = 0; q < ER; ++q) {
                            v[q] = w == 0 ? (uint32_t)(rk[q] >> 32) : w == 1 ? (uint32_t)rk[q] : rh[q];
                            const uint32_t x = lane_in(m[q]) ? v[q] : 0u;
                            top = top > x ? top : x;
                        }
                        worst[w] = wave_max_u32(top);
#pragma unroll
                        for (int q = 0; q < ER; ++q) m[q] &= ballot64(v[q] == worst[w]);
                    }
                    const uint64_t wk = ((uint64_t)worst[0] << 32) | worst[1];
                    if (k > wk || (k == wk && h > worst[2])) continue;
#pragma unroll
                    for (int q = 0; q < ER; ++q)
                        if (m[q]) place = (uint32_t)q * 64u + (uint32_t)__builtin_ctzll(m[q]);
                } else {
                    ++c;
                }
#pragma unroll
                for (int q = 0; q < ER; ++q) {
                    const uint64_t here = ballot64((uint32_t)q * 64u + lane == place);
                    dirty[q] |= here;
                    if (lane_in(here)) {
                        rk[q] = k;
                        rh[q] = h;
#pragma unroll
                        for (uint32_t i = 0; i < kRhalfGroup; ++i) g[q][i] = ~0ull;
                    }
                }
                continue;
            }
#pragma unroll
            for (int q = 0; q < ER; ++q) {
                if (!hit[q]) continue;
                dirty[q] |= hit[q];
                if (!lane_in(hit[q])) continue;
                const uint64_t e0 = rk[q], e1 = g[q][0], e2 = g[q][1], e3 = g[q][2];
                const uint32_t t = (uint32_t)k;
                const bool s0 = (uint32_t)e0 == t, s1 = (uint32_t)e1 == t, s2 = (uint32_t)e2 == t, s3 = (uint32_t)e3 == t;
                if ((s0 && e0 <= k) || (s1 && e1 <= k) || (s2 && e2 <= k) || (s3 && e3 <= k)) continue;
                // without the target's worse key, then with the new one
                const bool p1 = s0 || s1, p2 = p1 || s2, p3 = p2 || s3;
                const uint64_t f0 = s0 ? e1 : e0, f1 = p1 ? e2 : e1, f2 = p2 ? e3 : e2, f3 = p3 ? ~0ull : e3;
                rk[q] = k < f0 ? k : f0;
                g[q][0] = k < f0 ? f0 : k < f1 ? k : f1;
                g[q][1] = A.quota < 2u ? ~0ull : k < f1 ? f1 : k < f2 ? k : f2;
                g[q][2] = A.quota < 3u ? ~0ull : k < f2 ? f2 : k < f3 ? k : f3;
            }
        }
        wait_loads();  // as in the merge: before the stores, which a wait in the next iteration would include
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            if (!dirty[q] || !lane_in(dirty[q])) continue;
            const uint64_t at = base + (uint32_t)q * 64u + lane;
            A.slot_keys[at] = rk[q];
            A.slot_hash[at] = (uint16_t)rh[q];
            if (c < A.l_max) {
#pragma unroll
                for (uint32_t j = 0; j < kRhalfGroup; ++j) A.grp_keys[at * kRhalfGroup + j] = g[q][j];
            }
        }
        if (lane == 0 && c != d0.c) A.slot_count[r0.src] = c;
        r0 = r1;
        r1 = r2;
        d0 = d1;
    }
}

// Segment workspace layout (nseg entries each unless noted): sort keys and
// values in / out (u32), run sources, lengths and starts (u32), the run count
// (one u32), the segment descriptors in sorted order (uint4), then the
// temporary of the radix sort / run-length encoding / scan.
struct SegWs {
    uint32_t *keys_in, *keys_out, *vals_in, *vals_out, *run_src, *run_len, *run_start, *num_runs;
    uint4 *sorted;
    void *temp;
    size_t temp_bytes;
};
size_t seg_align(size_t x) { return (x + 255) & ~(size_t)255; }
int key_bits(uint32_t num_points) {
    int b = 1;
    while (b < 32 && ((uint64_t)1 << b) <= num_points) ++b;  // keys go up to num_points (unused segments)
    return b;
}
size_t seg_temp(uint64_t nseg, uint32_t num_points) {
    size_t sort = 0, rle = 0, scan = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, sort, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                       (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)nseg, 0,
                                       key_bits(num_points));
    (void)hipcub::DeviceRunLengthEncode::Encode(nullptr, rle, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                          (uint32_t *)nullptr, (uint32_t *)nullptr, (int)nseg);
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, scan, (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)nseg);
    return sort > rle ? (sort > scan ? sort : scan) : (rle > scan ? rle : scan);
}
SegWs seg_ws_layout(void *base, uint64_t nseg, uint32_t num_points) {
    SegWs w{};
    char *p = static_cast<char *>(base);
    const size_t a = seg_align(nseg * 4);
    uint32_t **arr[7] = {&w.keys_in, &w.keys_out, &w.vals_in, &w.vals_out, &w.run_src, &w.run_len, &w.run_start};
    for (int i = 0; i < 7; ++i) *arr[i] = reinterpret_cast<uint32_t *>(p + i * a);
    w.num_runs = reinterpret_cast<uint32_t *>(p + 7 * a);
    w.sorted = reinterpret_cast<uint4 *>(p + 7 * a + 256);
    w.temp = p + 7 * a + 256 + seg_align(nseg * 16);
    w.temp_bytes = seg_temp(nseg, num_points);
    return w;
}

// One wave per point: its slots sorted by hash (a reservoir's hashes are
// distinct, so the order is the reference's emit order, ascending hash).  The
// sort's exchanges bound it while they carried hash and key through LDS
// permutes: 524,288 points of 64 slots 378 us, one word through row moves 147
// (4.6 TB/s).
template <int ER>
__global__ __launch_bounds__(kHpThreads) void hp_export_kernel(const uint64_t *slot_keys, const uint16_t *slot_hash,
                                                               const uint32_t *slot_count, uint32_t num_points,
                                                               uint32_t l_max, uint32_t *targets, uint16_t *hashes,
                                                               float *dists, uint32_t *counts) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * kHpWaves;
    for (uint32_t p = blockIdx.x * kHpWaves + (threadIdx.x >> 6); p < num_points; p += waves) {
        const uint32_t c = slot_count[p];
        const uint64_t base = (uint64_t)p * l_max;
        uint32_t h[ER];
        uint64_t k[ER];
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const uint32_t e = (uint32_t)q * 64u + lane;
            h[q] = e < c ? (uint32_t)slot_hash[base + e] : 0xffffffffu;
            k[q] = e < c ? slot_keys[base + e] : ~0ull;
        }
        sort_slots<ER>(h, k, lane);
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const uint32_t e = (uint32_t)q * 64u + lane;
            if (e >= l_max) continue;
            const bool live = e < c;
            if (targets) targets[base + e] = live ? (uint32_t)k[q] : 0xffffffffu;
            if (hashes) hashes[base + e] = live ? (uint16_t)h[q] : (uint16_t)0;
            if (dists) dists[base + e] = live ? key_dist((uint32_t)(k[q] >> 32)) : 0.0f;
        }
        if (counts && lane == 0) counts[p] = c;
    }
}

// ---- named R-half backfill ----------------------------------------------------
// The reference's order-independent characterization of its R-half streaming
// reservoir (shear-core/src/algorithm/pipnn/hash_prune.rs:2601-2682
// reference_tiered_rhalf_slots; ranking :655-685, capacities
// hash_prune_backfill.rs:299-336, SoftTier score :375-386): a row with some
// but fewer than l_max primaries is completed with up to `capacity` backups,
// chosen by the mode's priority among each primary hash's next `quota`
// distinct targets (each at its best key, the primary's own target
// excluded; a member's hit layer is its rank in its group).
//
// Each slot keeps its hash's best quota + 1 distinct targets: the slot key and
// a group of quota keys.  That set does not depend on the order of the
// candidates (a target dropped from it had quota + 1 better distinct targets
// of the hash, whose keys only improve), so batches still merge in any
// order.  A reservoir that has filled never frees a slot and a full row takes
// no backups, so groups are kept only while a slot is free: hp_absorb merges a
// batch with its groups (quota + 1 rounds of best_of_hash), hp_few_kernel
// inserts a source's few records one by one.  Once the reservoir is full its
// slots are kept as without a policy, and the groups are neither read nor
// written again.  Slots lie in no particular order; the export ranks them.

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
    const uint32_t lo = __shfl_xor((uint32_t)v, m);
    const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), m);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t total_key64(double d) {
    const uint64_t b = (uint64_t)__double_as_longlong(d);
    return (b & 0x8000000000000000ull) ? ~b : (b | 0x8000000000000000ull);
}

// A group member's rank under the mode's priority (hash_prune.rs:655-685) as
// a 128-bit key (hi, lo); members are distinct (hash, target) pairs, so keys
// are distinct.  SoftTier: (score, layer, target, hash), the score the f64
// distance times alpha^2 per layer past the first (hash_prune_backfill.rs:
// 375-386); HardTier: (layer, distance, target, hash); the others:
// (distance, layer, target, hash).
__device__ __forceinline__ void member_rank(uint32_t mode, double alpha_sq, uint64_t key, uint32_t hash,
                                            uint32_t layer, uint64_t &hi, uint64_t &lo) {
    const uint32_t dk = (uint32_t)(key >> 32);
    const uint64_t th = ((uint64_t)(uint32_t)key << 16) | hash;
    if (mode == kRhalfSoftTierQ3) {
        double s = (double)key_dist(dk);
        if (layer >= 2) s = s * alpha_sq;
        if (layer >= 3) s = s * alpha_sq;
        hi = total_key64(s);
        lo = ((uint64_t)layer << 48) | th;
    } else if (mode == kRhalfHardTierQ3) {
        hi = ((uint64_t)layer << 32) | dk;
        lo = th;
    } else {
        hi = dk;
        lo = ((uint64_t)layer << 48) | th;
    }
}

// hp_export_kernel followed, for a row with some but fewer than l_max
// primaries, by min(capacity, l_max - c) backups: the best group members by
// the mode's priority, one wave-wide arg-min per backup, written after the
// primaries in priority order.
template <int ER>
__global__ __launch_bounds__(kHpThreads) void hp_export_rhalf_kernel(
    const uint64_t *slot_keys, const uint16_t *slot_hash, const uint32_t *slot_count, const uint64_t *grp_keys,
    uint32_t num_points, uint32_t l_max, uint32_t mode, uint32_t quota, uint32_t capacity, double alpha_sq,
    uint32_t *targets, uint16_t *hashes, float *dists, uint32_t *counts) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * kHpWaves;
    for (uint32_t p = blockIdx.x * kHpWaves + (threadIdx.x >> 6); p < num_points; p += waves) {
        const uint32_t c = slot_count[p];
        const uint64_t base = (uint64_t)p * l_max;
        uint32_t h[ER];
        uint64_t k[ER];
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const uint32_t e = (uint32_t)q * 64u + lane;
            h[q] = e < c ? (uint32_t)slot_hash[base + e] : 0xffffffffu;
            k[q] = e < c ? slot_keys[base + e] : ~0ull;
        }
        uint32_t take = 0;
        if (c > 0 && c < l_max) {
            const uint32_t cap = capacity < l_max - c ? capacity : l_max - c;
            uint64_t mh[ER][kRhalfGroup], ml[ER][kRhalfGroup];
#pragma unroll
            for (int q = 0; q < ER; ++q) {
                const uint32_t e = (uint32_t)q * 64u + lane;
#pragma unroll
                for (uint32_t j = 0; j < kRhalfGroup; ++j) {
                    const uint64_t g = e < c && j < quota ? grp_keys[(base + e) * kRhalfGroup + j] : ~0ull;
                    mh[q][j] = ~0ull;
                    ml[q][j] = ~0ull;
                    if (g != ~0ull) member_rank(mode, alpha_sq, g, h[q], j + 1u, mh[q][j], ml[q][j]);
                }
            }
            for (; take < cap; ++take) {
                uint64_t bh = ~0ull, bl = ~0ull;
                uint32_t bi = 0;
#pragma unroll
                for (int q = 0; q < ER; ++q) {
#pragma unroll
                    for (uint32_t j = 0; j < kRhalfGroup; ++j) {
                        const bool lt = mh[q][j] < bh || (mh[q][j] == bh && ml[q][j] < bl);
                        bh = lt ? mh[q][j] : bh;
                        bl = lt ? ml[q][j] : bl;
                        bi = lt ? (uint32_t)q * kRhalfGroup + j : bi;
                    }
                }
                uint64_t wh = bh, wl = bl;
#pragma unroll
                for (int m = 1; m < 64; m <<= 1) {
                    const uint64_t oh = shfl_xor64(wh, m), ol = shfl_xor64(wl, m);
                    const bool lt = oh < wh || (oh == wh && ol < wl);
                    wh = lt ? oh : wh;
                    wl = lt ? ol : wl;
                }
                if (wl == ~0ull) break;  // no member left (valid ranks never have lo = ~0)
                if (bh == wh && bl == wl) {
                    const uint64_t o = base + c + take;
#pragma unroll
                    for (int q = 0; q < ER; ++q) {
#pragma unroll
                        for (uint32_t j = 0; j < kRhalfGroup; ++j) {
                            if (bi != (uint32_t)q * kRhalfGroup + j) continue;
                            const uint64_t g = grp_keys[(base + (uint32_t)q * 64u + lane) * kRhalfGroup + j];
                            if (targets) targets[o] = (uint32_t)g;
                            if (hashes) hashes[o] = (uint16_t)h[q];
                            if (dists) dists[o] = key_dist((uint32_t)(g >> 32));
                            mh[q][j] = ~0ull;
                            ml[q][j] = ~0ull;
                        }
                    }
                }
            }
        }
        sort_slots<ER>(h, k, lane);
#pragma unroll
        for (int q = 0; q < ER; ++q) {
            const uint32_t e = (uint32_t)q * 64u + lane;
            if (e >= l_max || (e >= c && e < c + take)) continue;  // the backups' positions
            const bool live = e < c;
            if (targets) targets[base + e] = live ? (uint32_t)k[q] : 0xffffffffu;
            if (hashes) hashes[base + e] = live ? (uint16_t)h[q] : (uint16_t)0;
            if (dists) dists[base + e] = live ? key_dist((uint32_t)(k[q] >> 32)) : 0.0f;
        }
        if (counts && lane == 0) counts[p] = c + take;
    }
}

template <int ER>
void launch_few(const HpMergeArgs &A, uint32_t capacity, uint32_t grid, hipStream_t stream) {
    hipLaunchKernelGGL(hp_few_kernel<ER>, dim3(grid), dim3(kHpThreads), 0, stream, A, capacity);
}

template <int ER, bool kGrouped>
void launch_merge_er(const HpMergeArgs &A, bool rhalf, uint32_t grid, hipStream_t stream) {
    if (rhalf)
        hipLaunchKernelGGL((hp_merge_kernel<ER, true, kGrouped>), dim3(grid), dim3(kHpThreads), 0, stream, A);
    else
        hipLaunchKernelGGL((hp_merge_kernel<ER, false, kGrouped>), dim3(grid), dim3(kHpThreads), 0, stream, A);
}
template <bool kGrouped>
void launch_merge(const HpMergeArgs &A, bool rhalf, uint32_t grid, hipStream_t stream) {
    if (A.l_max <= 64)
        launch_merge_er<1, kGrouped>(A, rhalf, grid, stream);
    else if (A.l_max <= 128)
        launch_merge_er<2, kGrouped>(A, rhalf, grid, stream);
    else
        launch_merge_er<4, kGrouped>(A, rhalf, grid, stream);
}

uint32_t grid_for(uint64_t n, uint32_t threads, uint32_t cap) {
    const uint64_t g = (n + threads - 1) / threads;
    return (uint32_t)(g < 1 ? 1 : (g > cap ? cap : g));
}

}  // namespace

uint64_t hashprune_scan_blocks(uint32_t num_points) { return (num_points + kScanBlock - 1) / kScanBlock + 1; }

int launch_hashprune_clear(HashPruneState &s, hipStream_t stream) {
    hipLaunchKernelGGL(hp_fill_u32, dim3(grid_for(s.num_points, 256, 4096)), dim3(256), 0, stream, s.slot_count,
                       (uint64_t)s.num_points, 0u);
    hipLaunchKernelGGL(hp_fill_u32, dim3(grid_for(s.num_points, 256, 4096)), dim3(256), 0, stream, s.bucket,
                       (uint64_t)s.num_points, 0u);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_hashprune_insert(HashPruneState &s, const uint4 *records, uint64_t count, hipStream_t stream) {
    const uint32_t n = s.num_points;
    hipLaunchKernelGGL(hp_status_init, dim3(1), dim3(1), 0, stream, s.status);
    if (count == 0 || n == 0) return hipGetLastError() == hipSuccess ? 0 : -1;
    hipLaunchKernelGGL(hp_count_kernel, dim3(grid_for(count, 256, 16384)), dim3(256), 0, stream, records, count, n,
                       s.bucket, s.status);
    const uint32_t nb = (n + kScanBlock - 1) / kScanBlock;
    const HpRuns runs = record_runs(s);
    hipLaunchKernelGGL(hp_scan_reduce, dim3(nb), dim3(kScanThreads), 0, stream, s.bucket, n, s.block_sums);
    hipLaunchKernelGGL(hp_scan_partials, dim3(1), dim3(kScanThreads), 0, stream, s.block_sums, nb, s.offsets, n);
    hipLaunchKernelGGL(hp_scan_apply, dim3(nb), dim3(kScanThreads), 0, stream, s.bucket, n, s.block_sums, s.offsets, runs);
    hipLaunchKernelGGL(hp_scatter_kernel, dim3(grid_for(count, 256, 16384)), dim3(256), 0, stream, records, count, n,
                       s.bucket, s.offsets, s.grouped);
    const HpMergeArgs A{s.grouped, nullptr, runs.src, runs.start, runs.len, runs.count, n, s.l_max, s.rhalf_quota,
                        s.slot_keys, s.slot_hash, s.slot_count, s.grp_keys};
    const uint32_t grid = grid_for(count < n ? count : n, kHpWaves, kHpMergeGrid);
    if (runs.few) {
        if (s.l_max <= 64)
            launch_few<1>(A, runs.capacity, grid, stream);
        else if (s.l_max <= 128)
            launch_few<2>(A, runs.capacity, grid, stream);
        else
            launch_few<4>(A, runs.capacity, grid, stream);
    }
    launch_merge<true>(A, s.rhalf_mode != 0, grid, stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

uint64_t hashprune_segment_workspace_bytes(uint64_t nseg, uint32_t num_points) {
    const uint64_t n = nseg ? nseg : 1;
    return 7 * seg_align(n * 4) + 256 + seg_align(n * 16) + seg_temp(n, num_points) + 256;
}

int launch_hashprune_insert_segments(HashPruneState &s, const uint4 *records, const uint4 *segs, uint64_t nseg,
                                     hipStream_t stream) {
    const uint32_t n = s.num_points;
    hipLaunchKernelGGL(hp_status_init, dim3(1), dim3(1), 0, stream, s.status);
    if (nseg == 0 || n == 0) return hipGetLastError() == hipSuccess ? 0 : -1;
    SegWs w = seg_ws_layout(s.seg_ws, nseg, n);
    hipLaunchKernelGGL(hp_seg_keys_kernel, dim3(grid_for(nseg, 256, 16384)), dim3(256), 0, stream, segs, nseg, n,
                       w.keys_in, w.vals_in, s.status);
    size_t tb = w.temp_bytes;
    if (hipcub::DeviceRadixSort::SortPairs(w.temp, tb, w.keys_in, w.keys_out, w.vals_in, w.vals_out, (int)nseg, 0,
                                           key_bits(n), stream) != hipSuccess)
        return -1;
    tb = w.temp_bytes;
    if (hipcub::DeviceRunLengthEncode::Encode(w.temp, tb, w.keys_out, w.run_src, w.run_len, w.num_runs, (int)nseg,
                                              stream) != hipSuccess)
        return -1;
    // run starts: exclusive sum of the lengths (entries past the run count
    // are never read)
    tb = w.temp_bytes;
    if (hipcub::DeviceScan::ExclusiveSum(w.temp, tb, w.run_len, w.run_start, (int)nseg, stream) != hipSuccess)
        return -1;
    hipLaunchKernelGGL(hp_seg_gather_kernel, dim3(grid_for(nseg, 256, 16384)), dim3(256), 0, stream, segs,
                       w.vals_out, nseg, w.sorted);
    const HpMergeArgs A{records, w.sorted, w.run_src, w.run_start, w.run_len, w.num_runs, n, s.l_max,
                        s.rhalf_quota, s.slot_keys, s.slot_hash, s.slot_count, s.grp_keys};
    launch_merge<false>(A, s.rhalf_mode != 0, grid_for(nseg, kHpWaves, kHpMergeGrid), stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_hashprune_export(const HashPruneState &s, uint32_t *targets, uint16_t *hashes, float *dists,
                            uint32_t *counts, hipStream_t stream) {
    const uint32_t n = s.num_points;
    if (n == 0 || s.l_max == 0) return 0;
    const uint32_t grid = grid_for(n, kHpWaves, 8192);
    if (s.rhalf_mode) {
        if (s.l_max <= 64)
            hipLaunchKernelGGL(hp_export_rhalf_kernel<1>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys,
                               s.slot_hash, s.slot_count, s.grp_keys, n, s.l_max, s.rhalf_mode, s.rhalf_quota,
                               s.rhalf_capacity, s.rhalf_alpha_sq, targets, hashes, dists, counts);
        else if (s.l_max <= 128)
            hipLaunchKernelGGL(hp_export_rhalf_kernel<2>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys,
                               s.slot_hash, s.slot_count, s.grp_keys, n, s.l_max, s.rhalf_mode, s.rhalf_quota,
                               s.rhalf_capacity, s.rhalf_alpha_sq, targets, hashes, dists, counts);
        else
            hipLaunchKernelGGL(hp_export_rhalf_kernel<4>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys,
                               s.slot_hash, s.slot_count, s.grp_keys, n, s.l_max, s.rhalf_mode, s.rhalf_quota,
                               s.rhalf_capacity, s.rhalf_alpha_sq, targets, hashes, dists, counts);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    if (s.l_max <= 64)
        hipLaunchKernelGGL(hp_export_kernel<1>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys, s.slot_hash,
                           s.slot_count, n, s.l_max, targets, hashes, dists, counts);
    else if (s.l_max <= 128)
        hipLaunchKernelGGL(hp_export_kernel<2>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys, s.slot_hash,
                           s.slot_count, n, s.l_max, targets, hashes, dists, counts);
    else
        hipLaunchKernelGGL(hp_export_kernel<4>, dim3(grid), dim3(kHpThreads), 0, stream, s.slot_keys, s.slot_hash,
                           s.slot_count, n, s.l_max, targets, hashes, dists, counts);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tessa
