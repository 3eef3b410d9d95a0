// search.hip -- greedy search of a neighbour graph: the recall harness's
// search, one wavefront per query.
//
// Reference (paths relative to shear-core/src/): algorithm/search/search.rs:
// 137-233 (seed the list with the start point, mark it visited; repeatedly
// expand the closest not-visited entry; its unvisited neighbours are marked
// and inserted; stop when every listed entry is visited) over the capacity-L
// queue of model/neighbor/neighbor_priority_queue.rs:50-85, ordered by
// (distance, id) (model/neighbor/neighbor.rs:46-70); results as
// index/inmem_index/inmem_index.rs:559-580 (the first K entries).
//
// Inserting one expansion's neighbours one by one into the capacity-L sorted
// list leaves the L smallest of (list, neighbours) under the total order
// (distance, id), and the queue's cursor is then the first not-visited entry
// (an insert in front of the cursor moves it there; entries before it are all
// visited).  So the wave inserts the up-to-64 new neighbours of a chunk of the
// row at once, each entry going to its old place plus the number of entries of
// the other side below it; entries placed L and past drop off.  Same list,
// same cursor as the one-by-one inserts.
//
// Distances: squared L2 summed over the coordinates in order in f32, each
// product rounded before the add (no contraction), one lane per candidate
// (the harness's stated order; the reference's SIMD kernel may associate
// differently).  With SQ8 rows (sets too large to keep as f32) a row's
// coordinate i is the f32 product scale * code[i], rounded, then the same sum:
// the search over the dequantized vectors.  Keys are (distance bits << 32 |
// id): for the non-negative distances this computes, the integer order is
// (distance, id).
//
// Visited set: a bit per (slot, point), set by an atomic or, so a point listed
// twice in one row enters the list once; zeroed once per call, and by the
// slot's wave before its next query.
//
// The kernel waits, it does not compute: one wavefront per query and a chain of
// about L + 10 expansions, each of them neighbour ids -> visited bits -> rows ->
// distances -> list.  What it does about that:
//  * each lane reads its own row with 64 bytes or more in flight (direct_dist);
//    wide rows of few queries go to LDS instead (launch_graph_search: the rule
//    and both sides), by LDS-DMA, whole pieces by consecutive lanes and all in
//    flight together with the visited bits' atomics (the rows of neighbours that
//    turn out visited are read for nothing); one lane then sums one row from LDS;
//  * the neighbour ids of the entry that is next in line so far are read
//    meanwhile;
//  * the list is held in registers, and a pass over the new neighbours that can
//    still enter it gives every position by counting, without sorting;
//  * the visited set is one bit per point (25 KB per query at 200,000 points,
//    in L2) instead of a 4-byte tag: no 0.14 ms to clear 800 MB, and 32 times
//    the queries at a time on a set whose tags fill the scratch limit.
// 40,000 points, L = 64, against tags, a list in LDS and 16 to 32 bytes of a row
// in flight: 1,000 queries of 128 f32 columns 956 -> 530 us, of 768 4,364 -> 2,290;
// 4,000 queries of 256 SQ8 columns 1,799 -> 1,370; 20,000 of 97 f32 columns 13.0 ->
// 3.0 ms.
#include "search_kernels.h"
#include "tessa_device.h"
#include "kernel_attr.h"

namespace tessa {

namespace {

constexpr uint64_t kNoKey = ~0ull;

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ uint32_t readlane32(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ uint64_t readlane64(uint64_t v, uint32_t l) {
    return ((uint64_t)readlane32((uint32_t)(v >> 32), l) << 32) | readlane32((uint32_t)v, l);
}

// One more coordinate of a squared L2 distance, in order.
__device__ __forceinline__ float l2_step(float s, float x, float q) {
    const float t = __fsub_rn(x, q);
    return __fadd_rn(s, __fmul_rn(t, t));
}

// What the rows are.
enum SearchRows : int {
    kRowsF32 = 0,     // f32; staged: 16-byte aligned rows of dim % 4 == 0
    kRowsSq8x16 = 1,  // SQ8, 16-byte aligned rows
    kRowsSq8 = 2      // SQ8, any (not staged)
};

// Staged rows: columns (the query lies in LDS too), and the bytes of a row in
// LDS at a time (handed to the kernel: as a constant in it, the loops compile to
// something 3 % slower over f32 rows).
constexpr uint32_t kStagedMinF32 = 128, kStagedMinSq8 = 257, kStagedMaxDim = 2048;
constexpr uint32_t kStagedBytes = 512;

// LDS of a query's wave: staged rows' query (dim floats), the new list's keys
// and visited flags, staged rows.
struct SearchLds {
    uint32_t keys, flags, rows, row_stride, cols, bytes;  // byte offsets; columns of a row at a time
};
__host__ __device__ inline SearchLds search_lds(uint32_t dim, uint32_t L, int rows, bool staged, uint32_t row_bytes) {
    SearchLds s;
    s.keys = staged ? (dim + 3u) / 4u * 16u : 0u;
    s.flags = s.keys + L * 8u;
    s.rows = (s.flags + L * 4u + 15u) & ~15u;
    s.cols = rows == kRowsF32 ? (dim < row_bytes / 4u ? dim : row_bytes / 4u) : row_bytes;
    s.row_stride = (rows == kRowsF32 ? s.cols * 4u : s.cols) + 16u;  // the row lanes read different banks
    s.bytes = s.rows + (staged ? 64u * s.row_stride : 0u);
    return s;
}

// A lane's distance, the row read from memory (rows not staged).  64 lanes read
// 64 rows, so what a lane has in flight is what hides the latency, and a line
// read in several turns is gone from the L1 in between: 64 bytes of the row at a
// time, SQ8 rows (whose conversions take longer) with the next 64 on their way.
// The query is the wave's own and comes by scalar loads, which the rows' loads
// do not wait for.  1,000 queries, 40,000 points, L = 64: 4,096 SQ8 columns 11.2
// ms (32 bytes at a time and the query by vector loads 11.5, a byte at a time 4.5
// times that); 2,049 f32 columns, rows at any float's address, 7.2 ms (a float at
// a time 52).
template <int kRows>
__device__ __forceinline__ float direct_dist(const GraphSearchParams &p, uint32_t id, const float *query) {
    const auto *q = (const __attribute__((address_space(4))) float *)(uintptr_t)query;
    float s = 0.0f;
    uint32_t i = 0;
    if constexpr (kRows == kRowsF32) {
        typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
        const float *x = p.data + (uint64_t)id * p.dim;
        for (; i + 16u <= p.dim; i += 16u) {
            f4 a[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = reinterpret_cast<const f4 *>(x + i)[e];
#pragma unroll
            for (int e = 0; e < 16; ++e) s = l2_step(s, a[e / 4][e % 4], q[i + e]);
        }
        for (; i < p.dim; ++i) s = l2_step(s, x[i], q[i]);
    } else {
        const int8_t *c = p.codes + (uint64_t)id * p.padded_dim;
        const float sc = p.scales[id];
        if constexpr (kRows == kRowsSq8x16) {
            auto step = [&](const uint4 &w, uint32_t at) {
                const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    s = l2_step(s, __fmul_rn(sc, (float)(int8_t)(ww[e / 4] >> (8 * (e % 4)))), q[at + e]);
            };
            const uint4 *c16 = reinterpret_cast<const uint4 *>(c);
            const uint32_t turns = p.dim / 64u;
            if (turns) {
                uint4 w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = c16[e];
                for (uint32_t t = 0; t < turns; ++t) {
                    uint4 next[4];
                    const uint32_t u = t + 1u < turns ? t + 1u : t;
#pragma unroll
                    for (int e = 0; e < 4; ++e) next[e] = c16[4u * u + e];
#pragma unroll
                    for (int e = 0; e < 4; ++e) step(w[e], 64u * t + 16u * e);
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = next[e];
                }
                i = turns * 64u;
            }
            for (; i + 16u <= p.dim; i += 16u) step(c16[i / 16u], i);
        }
        for (; i < p.dim; ++i) s = l2_step(s, __fmul_rn(sc, (float)c[i]), q[i]);
    }
    return s;
}

// E: list entries per lane (entry e * 64 + lane), L <= 64 * E.  Rows not staged:
// registers for the four waves per SIMD that 4,096 slots make (with 130 instead
// of 128 registers, 20,000 queries over 768 SQ8 columns took 17.2 ms, not 14.2).
template <int kRows, bool kStaged, int E>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kStaged ? 0 : 4))) void graph_search_kernel(
    GraphSearchParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const SearchLds o = search_lds(p.dim, p.L, kRows, kStaged, p.row_bytes);
    float *ql = reinterpret_cast<float *>(lds);
    uint64_t *skey = reinterpret_cast<uint64_t *>(lds + o.keys);
    uint32_t *sflag = reinterpret_cast<uint32_t *>(lds + o.flags);
    unsigned char *rows = lds + o.rows;
    const uint32_t lane = threadIdx.x;
    const uint32_t words = search_words(p.num_points);
    uint32_t *seen = p.visited + (uint64_t)blockIdx.x * words;
    uint32_t pre_node = 0, pre_id = 0, pre_cnt = 0;  // neighbour ids read ahead
    bool pre = false;

    // neighbours [s0, s0 + 64) of a node (the ids past its degree are read too, where the row has them)
    auto load_ids = [&](uint32_t node, uint32_t s0) -> uint32_t {
        return s0 + lane < p.row_stride ? p.targets[(uint64_t)node * p.row_stride + s0 + lane] : 0xFFFFFFFFu;
    };

    // Marks the valid lanes' ids as visited; returns the lanes that were not
    // yet, with their distance in d.  next: a node whose ids are read ahead.
    auto score = [&](uint64_t valid, uint32_t id, const float *q, float &d, bool ahead, uint32_t next) -> uint64_t {
        const bool mine = (valid >> lane) & 1ull;
        uint32_t old = ~0u;
        if (mine) old = atomicOr(&seen[id >> 5], 1u << (id & 31u));
        uint64_t fresh = 0;
        float s = 0.0f, sc = 0.0f;
        auto claim = [&]() {
            uint32_t was = old;
            asm volatile("" : "+v"(was));  // keeps the test, and the wait for the atomic, here: behind the rows' loads
            fresh = __ballot(mine && !((was >> (id & 31u)) & 1u));
        };
        auto read_ahead = [&]() {
            if (ahead) {
                pre_cnt = p.counts[next];
                pre_id = load_ids(next, 0u);
            }
        };
        if constexpr (!kStaged) {
            read_ahead();
            claim();
            if ((fresh >> lane) & 1ull) s = direct_dist<kRows>(p, id, q);
        } else {
            using lds_ptr = __attribute__((address_space(3))) void *;
            if (kRows == kRowsSq8x16 && mine) sc = p.scales[id];
            uint64_t at = kRows == kRowsSq8x16 ? reinterpret_cast<uint64_t>(p.codes) + (uint64_t)id * p.padded_dim
                                               : reinterpret_cast<uint64_t>(p.data) + (uint64_t)id * p.dim * 4u;
            asm volatile("" : "+v"(at));  // all 64 lanes have their address before the branch that reads it by lane
            auto stage = [&](uint32_t c0, uint32_t n, uint64_t m) __attribute__((always_inline)) {
                wave_lds_sync();
                __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): what lies in the rows' place has been read
                // Row j's address by two lane reads.  Nearly all rows of a
                // full chunk: an unrolled loop over all 64 (the others read
                // row 0), half the instructions of walking the mask.
                auto each = [&](auto &&dma) {
                    auto one = [&](uint32_t j) {
                        dma(reinterpret_cast<const unsigned char *>(readlane64(at, j)) + c0 * (kRows == kRowsSq8x16 ? 1u : 4u),
                            rows + j * o.row_stride);
                    };
                    if (__popcll(m) > 48) {
#pragma unroll 8
                        for (uint32_t j = 0; j < 64u; ++j) one(j);
                    } else {
                        for (; m; m &= m - 1ull) one((uint32_t)__builtin_ctzll(m));
                    }
                };
                // 16 bytes per lane, a row's piece of at most 512 bytes by 32 lanes
                const uint32_t bytes = kRows == kRowsF32 ? n * 4u : (n + 15u) & ~15u;
                if (lane * 16u < bytes)
                    each([&](const unsigned char *src, unsigned char *dst) {
                        __builtin_amdgcn_global_load_lds(static_cast<const void *>(src + lane * 16u), (lds_ptr)dst, 16, 0,
                                                         0);
                    });
            };
            auto landed = [&]() __attribute__((always_inline)) {
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the rows are in LDS
                wave_lds_sync();
            };
            auto sum = [&](uint32_t c0, uint32_t n) __attribute__((always_inline)) {
                const unsigned char *row = rows + lane * o.row_stride;
                if constexpr (kRows == kRowsF32) {
                    const float4 *x4 = reinterpret_cast<const float4 *>(row);
                    const float4 *q4 = reinterpret_cast<const float4 *>(ql + c0);
#pragma unroll 4
                    for (uint32_t t = 0; t < n / 4u; ++t) {
                        const float4 a = x4[t], b = q4[t];
                        s = l2_step(s, a.x, b.x);
                        s = l2_step(s, a.y, b.y);
                        s = l2_step(s, a.z, b.z);
                        s = l2_step(s, a.w, b.w);
                    }
                } else {
                    const int8_t *c = reinterpret_cast<const int8_t *>(row);
                    const uint4 *c16 = reinterpret_cast<const uint4 *>(row);
                    for (uint32_t t = 0; t < n / 16u; ++t) {
                        const uint4 w = c16[t];
                        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const float4 b = *reinterpret_cast<const float4 *>(ql + c0 + 16u * t + 4u * g);
                            const float bq[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                s = l2_step(s, __fmul_rn(sc, (float)(int8_t)(ww[g] >> (8 * e))), bq[e]);
                        }
                    }
                    for (uint32_t t = n & ~15u; t < n; ++t) s = l2_step(s, __fmul_rn(sc, (float)c[t]), ql[c0 + t]);
                }
            };
            // The first piece outside the loop: inside it, the compiler waits
            // for the atomic ahead of the loop, and the rows' loads after it.
            const uint32_t n0 = p.dim < o.cols ? p.dim : o.cols;
            stage(0u, n0, valid);
            read_ahead();
            landed();
            claim();
            if (fresh) {
                sum(0u, n0);
                for (uint32_t c0 = o.cols; c0 < p.dim; c0 += o.cols) {
                    const uint32_t n = p.dim - c0 < o.cols ? p.dim - c0 : o.cols;
                    stage(c0, n, fresh);
                    landed();
                    sum(c0, n);
                }
            }
        }
        d = s;
        return fresh;
    };

    for (uint32_t qi = blockIdx.x; qi < p.num_queries; qi += p.slots) {
        const float *q = p.queries + (uint64_t)qi * p.dim;
        if (qi != blockIdx.x) {
            // the slot's next query: its visited bits are cleared by its own wave
            uint4 *v = reinterpret_cast<uint4 *>(seen);
            for (uint32_t i = lane; i < words / 4u; i += 64u) v[i] = make_uint4(0u, 0u, 0u, 0u);
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): cleared before the atomics
            wave_lds_sync();
        }
        if constexpr (kStaged) {
            wave_lds_sync();
            for (uint32_t i = lane; i < p.dim; i += 64u) ql[i] = q[i];
            wave_lds_sync();
        }
        uint64_t lk[E];  // the list, ascending; kNoKey past its size
        bool open[E];    // entries not yet expanded
        uint32_t size = 1, cmps = 0;
        float d0;
        pre = false;
        score(1ull, p.start, q, d0, false, 0u);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            lk[e] = e == 0 && lane == 0 ? ((uint64_t)__float_as_uint(d0) << 32) | p.start : kNoKey;
            open[e] = e == 0 && lane == 0;
        }
        // the first open entry (closest_notvisited)
        auto first_open = [&](uint32_t &node) -> bool {
            bool any = false;
#pragma unroll
            for (int e = E - 1; e >= 0; --e) {
                const uint64_t m = __ballot(open[e]);
                if (m) {
                    node = readlane32((uint32_t)lk[e], (uint32_t)__builtin_ctzll(m));
                    any = true;
                }
            }
            return any;
        };
        uint32_t node = 0;
        while (first_open(node)) {
#pragma unroll
            for (int e = 0; e < E; ++e) open[e] = open[e] && (uint32_t)lk[e] != node;
            uint32_t next = 0;
            const bool ahead = first_open(next);
            const bool have = pre && pre_node == node;
            const uint32_t cnt = readlane32(have ? pre_cnt : p.counts[node], 0u);
            uint32_t ids = have ? pre_id : load_ids(node, 0u);
            pre = ahead;
            pre_node = next;
            const uint32_t deg = cnt < p.row_stride ? cnt : p.row_stride;
            for (uint32_t s0 = 0; s0 < deg; s0 += 64u) {
                if (s0) ids = load_ids(node, s0);
                const uint64_t valid = __ballot(s0 + lane < deg && ids < p.num_points);
                if (!valid) {
                    if (s0 == 0u) pre = false;  // nothing was read ahead
                    continue;
                }
                const uint32_t id = (valid >> lane) & 1ull ? ids : 0u;
                float d;
                const uint64_t fresh = score(valid, id, q, d, s0 == 0u && ahead, next);
                cmps += (uint32_t)__popcll(fresh);
                const uint64_t key = ((uint64_t)__float_as_uint(d) << 32) | id;
                // a full list takes what is better than its last entry
                uint64_t last = kNoKey;
                if (size == p.L) {
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        if ((p.L - 1u) / 64u == (uint32_t)e) last = readlane64(lk[e], (p.L - 1u) & 63u);
                }
                const uint64_t pass = fresh & __ballot(key < last || size < p.L);
                if (!pass) continue;
                // each passing key's place among them and in the list, each
                // entry's shift, by counting
                uint32_t place = 0, shift[E];
#pragma unroll
                for (int e = 0; e < E; ++e) shift[e] = 0;
                uint64_t m = pass;
                while (m) {
                    const uint32_t j = (uint32_t)__builtin_ctzll(m);
                    m &= m - 1ull;
                    const uint64_t kj = readlane64(key, j);
                    uint32_t under = 0;
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        const bool lt = lk[e] < kj;
                        under += (uint32_t)__popcll(__ballot(lt));
                        shift[e] += lt ? 0u : 1u;
                    }
                    place += kj < key ? 1u : 0u;
                    place += lane == j ? under : 0u;
                }
                wave_lds_sync();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const uint32_t at = (uint32_t)e * 64u + lane, pos = at + shift[e];
                    if (at < size && pos < p.L) {
                        skey[pos] = lk[e];
                        sflag[pos] = open[e] ? 1u : 0u;
                    }
                }
                if (((pass >> lane) & 1ull) && place < p.L) {
                    skey[place] = key;
                    sflag[place] = 1u;
                }
                const uint32_t grown = size + (uint32_t)__popcll(pass);
                size = grown < p.L ? grown : p.L;
                wave_lds_sync();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const uint32_t at = (uint32_t)e * 64u + lane;
                    lk[e] = kNoKey;
                    open[e] = false;
                    if (at < size) {
                        lk[e] = skey[at];
                        open[e] = sflag[at] != 0u;
                    }
                }
            }
            if (deg == 0u) pre = false;
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t i = (uint32_t)e * 64u + lane;
            if (i < p.K) {
                p.out_ids[(uint64_t)qi * p.K + i] = i < size ? (uint32_t)lk[e] : 0xFFFFFFFFu;
                if (p.out_dists)
                    p.out_dists[(uint64_t)qi * p.K + i] = i < size ? __uint_as_float((uint32_t)(lk[e] >> 32)) : 0.0f;
            }
        }
        if (p.out_cmps && lane == 0) p.out_cmps[qi] = cmps;
    }
}

__global__ void zero_words(uint4 *v, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        v[i] = make_uint4(0u, 0u, 0u, 0u);
}

template <int kRows, bool kStaged>
int launch_rows(const GraphSearchParams &p, hipStream_t stream) {
    const uint32_t bytes = search_lds(p.dim, p.L, kRows, kStaged, p.row_bytes).bytes;
    auto go = [&](auto kernel) -> int {
        if (ensure_lds_limit(reinterpret_cast<const void *>(kernel), (int)bytes)) return -1;
        hipLaunchKernelGGL(kernel, dim3(p.slots), dim3(64), bytes, stream, p);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    };
    if (p.L <= 64) return go(graph_search_kernel<kRows, kStaged, 1>);
    if (p.L <= 128) return go(graph_search_kernel<kRows, kStaged, 2>);
    return go(graph_search_kernel<kRows, kStaged, 4>);
}

}  // namespace

uint32_t search_slots(uint32_t num_points, uint32_t num_queries) {
    // at most 1 GiB of visited bits and 4096 slots, at least one
    const uint64_t by_mem = (1ull << 30) / (4ull * search_words(num_points));
    uint64_t s = num_queries < 4096u ? num_queries : 4096u;
    if (s > by_mem) s = by_mem;
    return (uint32_t)(s < 1 ? 1 : s);
}

int launch_graph_search(const GraphSearchParams &params, hipStream_t stream) {
    GraphSearchParams p = params;
    p.row_bytes = kStagedBytes;
    const uint64_t n = (uint64_t)p.slots * search_words(p.num_points) / 4u;
    uint64_t zg = (n + 255) / 256;
    zg = zg < 1 ? 1 : (zg > 2048 ? 2048 : zg);
    hipLaunchKernelGGL(zero_words, dim3((uint32_t)zg), dim3(256), 0, stream, reinterpret_cast<uint4 *>(p.visited), n);
    auto aligned = [](const void *x) { return (reinterpret_cast<uintptr_t>(x) & 15u) == 0u; };
    // Rows are staged while every query has a SIMD to itself and all lie on the
    // chip at once.  Staged over read by the lanes, 16 to 1,000 queries: f32 rows
    // of 768 to 2,048 columns 0.83-1.08 of the time at L = 64 and 256 (1.05-1.3 at
    // 16), of 128 to 512 columns 0.89-1.1 with 1,000 queries (0.95 on 5,000,000
    // points) and 1.0-1.7 with few; SQ8 rows of 257 to 2,048 columns 0.84-1.16.
    // Narrower f32 rows take 0.98-1.4, narrower SQ8 rows 1.06-1.4.  With more
    // queries the rows of visited neighbours cost bandwidth and the LDS keeps
    // waves off the chip: 1,100 to 20,000 queries, in pieces of 512 or 256 bytes,
    // 0.98-1.8.  Rows at any float's address would be staged 4 bytes at a time:
    // 2.3-6.
    auto pays = [&](int rows) {
        const uint32_t per_cu = 160u * 1024u / search_lds(p.dim, p.L, rows, true, p.row_bytes).bytes;
        return p.dim >= (rows == kRowsF32 ? kStagedMinF32 : kStagedMinSq8) && p.dim <= kStagedMaxDim && p.slots <= 256u * per_cu;
    };
    if (p.data)
        return p.dim % 4u == 0u && aligned(p.data) && pays(kRowsF32) ? launch_rows<kRowsF32, true>(p, stream)
                                                                     : launch_rows<kRowsF32, false>(p, stream);
    if (p.padded_dim % 16u == 0u && aligned(p.codes))
        return pays(kRowsSq8x16) ? launch_rows<kRowsSq8x16, true>(p, stream)
                                 : launch_rows<kRowsSq8x16, false>(p, stream);
    return launch_rows<kRowsSq8, false>(p, stream);
}

}  // namespace tessa
