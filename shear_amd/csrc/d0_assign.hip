// d0_assign.hip -- global D0 assignment on gfx950 int8 MFMA: every SQ8 row
// to its fanout_top (<= 32) nearest global D0 leaders, then the fragments
// grouped into the D0 children.
//
// Reference (shear-core/src/algorithm/pipnn/compute_backend.rs): the GPU-D0
// kernels sq8_global_d0_tiled_partial_kernel / sq8_global_d0_wmma_partial_kernel
// (:18016-18275, per leader tile the best partial_r leaders of each row) and
// the merge rabitq_residual_global_d0_tiled_merge_kernel (:18446-18511, the
// best fanout_top over the tiles), both ordered by (dist, leader global id)
// strictly, the distance sq_int8_approx_l2 (dco_sq_int8.rs:2950-2965):
// (norm_r + norm_l) - ((2 * scale_r) * scale_l) * dot, clamped at 0.  Output
// fragments row-major (child = leader index, point = global id, :18503-18510).
//
// Here one pass replaces partial + merge: a wave holds 32 rows' codes in VGPRs
// as the MFMA B operand and streams the leaders 32 at a time as A.  The eight
// waves of a workgroup (256 rows) share each leader tile through LDS (double
// buffered; the next tile's codes, scales, norms and ranks are loaded into
// registers while the current one is used), so a tile crosses L2 once per
// 256 rows instead of once per 32; each lane owns one row and
// half of a tile's leaders and keeps its best F >= fanout (distance bits << 32
// | leader rank) keys sorted in registers, inserting a candidate only when it
// beats the current F-th.  The two halves of a row merge at the end.  A
// leader's rank is its position in (leader id, index) order, so the key's
// integer order is the reference's order (distances are >= 0).
//
// Bound: MFMA, LDS reads (a leader fragment per MFMA, as many LDS cycles as
// MFMA cycles) and the ranking added up, 2.72 ms for 2M rows x 768 and 1,000
// leaders (grouping included) where the products alone take 0.92.  For short
// lists d0_assign_wide_kernel halves the LDS reads and ranks during the MFMAs:
// 2.13 ms.
//
// Grouping: an LSD radix sort of (child, point) pairs by child, stable, so a
// child's points keep ascending row order; offsets from a child histogram.
#include <hipcub/hipcub.hpp>

#include "kernel_attr.h"
#include "d0_kernels.h"
#include "tessa_device.h"

namespace tessa {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8;  // 256 rows per workgroup share each leader tile
constexpr int kThreads = kWaves * 64;
constexpr uint32_t kWideLeaders = 128;  // more: the kernel with 64 rows per wave, for up to four per row
constexpr uint64_t kNoKey = ~0ull;
constexpr double kNoDKey = __builtin_inf();

// rank of each leader in (id, index) order; O(leaders^2) compares, leaders are few
__global__ void d0_rank_kernel(const uint32_t *ids, uint32_t n, uint32_t *rank, uint32_t *inv) {
    const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= n) return;
    const uint32_t me = ids[l];
    uint32_t r = 0;
    for (uint32_t o = 0; o < n; ++o) {
        const uint32_t v = ids[o];
        r += (v < me || (v == me && o < l)) ? 1u : 0u;
    }
    rank[l] = r;
    inv[r] = l;
}

template <int F>
__device__ __forceinline__ void insert_key(uint64_t (&best)[F], uint64_t key) {
#pragma unroll
    for (int s = 0; s < F; ++s) {
        const uint64_t b = best[s];
        const bool lt = key < b;
        best[s] = lt ? key : b;
        key = lt ? b : key;
    }
}

// merge the other half-wave's list into lanes 0..31 and write the row's fragments
template <int F>
__device__ __forceinline__ void write_best(const D0AssignParams &p, uint64_t (&best)[F], uint64_t row, uint32_t lane) {
    const uint32_t j = lane & 31u, h = lane >> 5;
#pragma unroll
    for (int s = 0; s < F; ++s) {
        const uint64_t o = ((uint64_t)__shfl((uint32_t)(best[s] >> 32), j + 32u) << 32) |
                           __shfl((uint32_t)best[s], j + 32u);
        if (h == 0u && o < best[F - 1]) insert_key<F>(best, o);
    }
    if (h == 0u && row < p.rows) {
        const uint32_t g = p.global_ids[row];
#pragma unroll
        for (int s = 0; s < F; ++s) {
            if ((uint32_t)s < p.fanout) {
                const uint32_t r = (uint32_t)best[s];  // always a real leader: fanout <= leaders
                p.out_child[row * p.fanout + s] = r < p.leaders ? p.rank_leader[r] : kEmptyId;
                p.out_point[row * p.fanout + s] = g;
            }
        }
    }
}

// v_min_f64 / v_max_f64 themselves: __builtin_fmin puts a v_max_f64(x, x) before
// each, which only a signalling NaN needs and no key is one.
__device__ __forceinline__ double min_f64(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ double max_f64(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Keys as doubles (see rank_key): ascending, branch-free for short lists
template <int F>
__device__ __forceinline__ void insert_key(double (&best)[F], double key) {
#pragma unroll
    for (int s = 0; s < F; ++s) {
        const double b = best[s];
        best[s] = min_f64(b, key);
        if (s + 1 < F) key = max_f64(b, key);
    }
}

// The key as a double: ascending doubles are ascending integers, v_min_f64 and
// v_max_f64 take one instruction each and keep subnormals.  A high word over
// 0x7fefffff would be a NaN or an infinity: only NaN distances have one, and the
// clamp leaves them behind every number.  ps2 = 2 * ps (rounded as in assign_l2);
// the IEEE maximum keeps a NaN, as assign_l2's compare does.
__device__ __forceinline__ double rank_key(int dot, float ps2, float pn, float ls, float ln, uint32_t rank) {
    const float c = __fmul_rn(__fmul_rn(ps2, ls), (float)dot);
    float d = __fsub_rn(__fadd_rn(pn, ln), c);
    d = __builtin_elementwise_maximum(d, 0.0f);
    const uint32_t hi = min(__float_as_uint(d), 0x7fefffffu);
    return __hiloint2double((int)hi, (int)rank);
}

template <int KS>
struct D0Tile {
    static constexpr int kStride = KS * 32 + 16;          // bytes per leader row (16-byte pad: no bank aliasing)
    static constexpr int kCodeBytes = 32 * kStride;
    static constexpr int kChunks = 32 * KS * 2;           // 16-byte chunks of the tile's codes
    static constexpr int kPerThread = (kChunks + kThreads - 1) / kThreads;
    static constexpr int kBytes = kCodeBytes + 32 * 12;  // + scales, norms, ranks
};

template <int KS, int F>
__global__ __launch_bounds__(kThreads) void d0_assign_kernel(D0AssignParams p) {
    using T = D0Tile<KS>;
    extern __shared__ __attribute__((aligned(16))) int8_t tiles[];  // 2 x T::kBytes
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t j = lane & 31u, h = lane >> 5;
    const uint64_t row = (uint64_t)blockIdx.x * (kWaves * 32) + wave * 32u + j;
    const bool ok = row < p.rows;
    const uint32_t pd = p.padded_dim;
    const uint32_t nl = p.leaders;

    v4i bfrag[KS];
    const int8_t *rc = p.codes + (ok ? row : 0ull) * pd;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const uint32_t off = 32u * s + 16u * h;
        v4i z = {0, 0, 0, 0};
        if (ok && off < pd) z = *reinterpret_cast<const v4i *>(rc + off);
        bfrag[s] = z;
    }
    const float rs = ok ? p.scales[row] : 0.0f;
    const float rn = ok ? p.norms[row] : 0.0f;

    uint64_t best[F];
#pragma unroll
    for (int s = 0; s < F; ++s) best[s] = kNoKey;

    // the next tile in registers: this thread's code chunks and one meta word
    v4i pre[T::kPerThread];
    uint32_t pmeta = 0u;
    auto issue = [&](uint32_t t) {
#pragma unroll
        for (int q = 0; q < T::kPerThread; ++q) {
            const uint32_t c = tid + (uint32_t)q * kThreads;
            const uint32_t li = c / (KS * 2), off = (c % (KS * 2)) * 16u;
            const uint32_t l = 32u * t + li;
            v4i z = {0, 0, 0, 0};
            if (c < (uint32_t)T::kChunks && l < nl && off < pd)
                z = *reinterpret_cast<const v4i *>(p.leader_codes + (uint64_t)l * pd + off);
            pre[q] = z;
        }
        if (tid < 96u) {
            const uint32_t l = 32u * t + (tid & 31u);
            const uint32_t li = l < nl ? l : 0u;
            pmeta = tid < 32u ? __float_as_uint(p.leader_scales[li])
                              : tid < 64u ? __float_as_uint(p.leader_norms[li]) : p.leader_rank[li];
        }
    };
    auto store = [&](int8_t *dst) {
#pragma unroll
        for (int q = 0; q < T::kPerThread; ++q) {
            const uint32_t c = tid + (uint32_t)q * kThreads;
            if (c < (uint32_t)T::kChunks) {
                const uint32_t li = c / (KS * 2), off = (c % (KS * 2)) * 16u;
                *reinterpret_cast<v4i *>(dst + li * T::kStride + off) = pre[q];
            }
        }
        if (tid < 96u) reinterpret_cast<uint32_t *>(dst + T::kCodeBytes)[tid] = pmeta;
    };

    const uint32_t ntiles = (nl + 31u) / 32u;
    issue(0);
    store(tiles);
    if (ntiles > 1u) issue(1);
    for (uint32_t t = 0; t < ntiles; ++t) {
        // tile t is in buffer t & 1; the other buffer was last read at t - 1
        __syncthreads();
        int8_t *cur = tiles + (t & 1u) * T::kBytes;
        if (t + 1u < ntiles) {
            store(tiles + ((t + 1u) & 1u) * T::kBytes);
            if (t + 2u < ntiles) issue(t + 2u);
        }
        const int8_t *arow = cur + j * T::kStride + 16u * h;
        v16i acc = {};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const v4i a = *reinterpret_cast<const v4i *>(arow + 32 * s);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, bfrag[s], acc, 0, 0, 0);
        }
        // lane value v is leader 8*(v/4) + 4h + v%4 of the tile: four consecutive
        // leaders per group, their scales / norms / ranks read as 16-byte vectors
        const float4 *tsc = reinterpret_cast<const float4 *>(cur + T::kCodeBytes);
        const float4 *tno = tsc + 8;
        const uint4 *trk = reinterpret_cast<const uint4 *>(tno + 8);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 sc4 = tsc[2 * g + h], no4 = tno[2 * g + h];
            const uint4 rk4 = trk[2 * g + h];
            const float scv[4] = {sc4.x, sc4.y, sc4.z, sc4.w}, nov[4] = {no4.x, no4.y, no4.z, no4.w};
            const uint32_t rkv[4] = {rk4.x, rk4.y, rk4.z, rk4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = 4 * g + e;
                const uint32_t l = 32u * t + 8u * g + 4u * h + e;
                const bool live = ok && l < nl;
                const float d = assign_l2(acc[v], rs, rn, scv[e], nov[e]);
                const uint64_t key = live ? (((uint64_t)__float_as_uint(d) << 32) | rkv[e]) : kNoKey;
                if (key < best[F - 1]) insert_key<F>(best, key);
            }
        }
    }
    write_best<F>(p, best, row, lane);
}

// The same assignment with 64 rows per wave, four waves (256 rows) per
// workgroup: a leader fragment read from LDS feeds two MFMAs, and the previous
// tile's distances are ranked between the MFMAs of the current one.  One wave per
// SIMD from 16 steps on: the rows' fragments alone are 2 * 4 * KS registers.
// What is left over the MFMAs' time is the ranking (about 11 VALU instructions
// per distance), and the load of the rows before the first tile.
constexpr int kWideWaves = 4;
constexpr int kWideThreads = kWideWaves * 64;

template <int KS>
struct D0WideTile {
    static constexpr int kStride = KS * 32 + 16;
    static constexpr int kCodeBytes = 32 * kStride;
    static constexpr int kPerThread = 32 * KS * 2 / kWideThreads;  // 16-byte chunks per thread, exact
    static constexpr int kMetaBytes = 32 * 12;                     // scales, norms, ranks
    static constexpr int kBytes = 2 * kCodeBytes + 3 * kMetaBytes;
    static_assert(32 * KS * 2 % kWideThreads == 0, "whole chunks per thread");
};

template <int KS, int F>
__global__ __launch_bounds__(kWideThreads, KS > 8 ? 1 : 2) void d0_assign_wide_kernel(D0AssignParams p) {
    using T = D0WideTile<KS>;
    extern __shared__ __attribute__((aligned(16))) int8_t tiles[];  // two code tiles, three tiles' meta words
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t j = lane & 31u, h = lane >> 5;
    const uint64_t row0 = (uint64_t)blockIdx.x * (kWideWaves * 64) + wave * 64u + j;
    const uint32_t pd = p.padded_dim;
    const uint32_t nl = p.leaders;

    // rows past the end take the last row's data; nothing is written for them
    v4i bfrag[2][KS];
    float rs[2], rn[2];
    double best[2][F];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint64_t row = row0 + 32u * r < p.rows ? row0 + 32u * r : p.rows - 1;
        const int8_t *rc = p.codes + row * pd;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const uint32_t off = 32u * s + 16u * h;
            v4i z = {0, 0, 0, 0};
            if (off < pd) z = *reinterpret_cast<const v4i *>(rc + off);
            bfrag[r][s] = z;
        }
        rs[r] = __fmul_rn(2.0f, p.scales[row]);
        rn[r] = p.norms[row];
#pragma unroll
        for (int s = 0; s < F; ++s) best[r][s] = kNoDKey;
    }

    // The next tile in registers.  Leaders past the end take the last one's
    // data (ranked by nobody); columns past the padding meet zeros in bfrag.
    v4i pre[T::kPerThread];
    uint32_t pmeta = 0u;
    auto issue = [&](int q, uint32_t t) {
        const uint32_t c = tid + (uint32_t)q * kWideThreads;
        const uint32_t l = min(32u * t + c / (KS * 2), nl - 1u), o = (c % (KS * 2)) * 16u;
        pre[q] = *reinterpret_cast<const v4i *>(p.leader_codes + (uint64_t)l * pd + (o < pd ? o : 0u));
    };
    auto store = [&](int q, uint32_t t) {
        const uint32_t c = tid + (uint32_t)q * kWideThreads;
        *reinterpret_cast<v4i *>(tiles + (t & 1u) * T::kCodeBytes + c / (KS * 2) * T::kStride + (c % (KS * 2)) * 16u) =
            pre[q];
    };
    const uint32_t *msrc = tid < 32u ? reinterpret_cast<const uint32_t *>(p.leader_scales)
                           : tid < 64u ? reinterpret_cast<const uint32_t *>(p.leader_norms) : p.leader_rank;
    auto issue_meta = [&](uint32_t t) { pmeta = msrc[min(32u * t + (tid & 31u), nl - 1u)]; };
    int8_t *const metas = tiles + 2 * T::kCodeBytes;
    auto store_meta = [&](uint32_t slot) {
        if (tid < 96u) reinterpret_cast<uint32_t *>(metas + slot * T::kMetaBytes)[tid] = pmeta;
    };
    // lane value v of a row group is leader 8*(v/4) + 4h + v%4 of the tile
    float4 sc4[4], no4[4];
    uint4 rk4[4];
    auto load_meta = [&](int g, uint32_t slot) {
        const float4 *m = reinterpret_cast<const float4 *>(metas + slot * T::kMetaBytes) + 2 * g + h;
        sc4[g] = m[0];
        no4[g] = m[8];
        rk4[g] = reinterpret_cast<const uint4 *>(m)[16];
    };
    auto rank_value = [&](int r, int v, int dot, bool live) {
        const float *sc = reinterpret_cast<const float *>(&sc4[v / 4]), *no = reinterpret_cast<const float *>(&no4[v / 4]);
        const uint32_t rk = reinterpret_cast<const uint32_t *>(&rk4[v / 4])[v % 4];
        const double key = rank_key(dot, rs[r], rn[r], sc[v % 4], no[v % 4], rk);
        insert_key<F>(best[r], live ? key : kNoDKey);
    };

    const uint32_t ntiles = (nl + 31u) / 32u;
#pragma unroll
    for (int q = 0; q < T::kPerThread; ++q) issue(q, 0);
    issue_meta(0);
#pragma unroll
    for (int q = 0; q < T::kPerThread; ++q) store(q, 0);
    store_meta(0);
#pragma unroll
    for (int q = 0; q < T::kPerThread; ++q) issue(q, 1);
    issue_meta(1);

    // nothing before tile 0: its keys are of NaN distances, behind every leader's
    if (tid < 96u) reinterpret_cast<uint32_t *>(metas + 2 * T::kMetaBytes)[tid] = 0x7fffffffu;
    v16i prev[2] = {};
    uint32_t slot = 0;  // t % 3
    for (uint32_t t = 0; t < ntiles; ++t) {
        // Tile t is in code buffer t & 1 and meta slot t % 3; the other buffer
        // was last read at t - 1, slot (t + 1) % 3 at t - 1 too (tile t - 2).
        __syncthreads();
        const uint32_t before = slot == 0u ? 2u : slot - 1u, after = slot == 2u ? 0u : slot + 1u;
        const int8_t *arow = tiles + (t & 1u) * T::kCodeBytes + j * T::kStride + 16u * h;
        constexpr int kAhead = 4;
        v4i a[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) a[s] = *reinterpret_cast<const v4i *>(arow + 32 * s);
#pragma unroll
        for (int g = 0; g < 4; ++g) load_meta(g, before);
        v16i acc[2] = {};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const v4i as = a[s % kAhead];
            if (s + kAhead < KS) a[s % kAhead] = *reinterpret_cast<const v4i *>(arow + 32 * (s + kAhead));
            acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(as, bfrag[0][s], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(as, bfrag[1][s], acc[1], 0, 0, 0);
            // the next tile to LDS and the one after it into registers
            if (s < T::kPerThread) {
                store(s, t + 1u);
                issue(s, t + 2u);
            }
            if (s == T::kPerThread) {
                store_meta(after);
                issue_meta(t + 2u);
            }
#pragma unroll
            for (int w = 32 * s / KS; w < 32 * (s + 1) / KS; ++w) {
                int dot = prev[w & 1][w >> 1];
                asm volatile("" : "+v"(dot));  // keeps the ranking in this step
                rank_value(w & 1, w >> 1, dot, true);
                asm volatile("" : "+v"(best[w & 1][F - 1]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        prev[0] = acc[0];
        prev[1] = acc[1];
        slot = after;
    }
    {
        const uint32_t last = slot == 0u ? 2u : slot - 1u;
#pragma unroll
        for (int g = 0; g < 4; ++g) load_meta(g, last);
#pragma unroll
        for (int w = 0; w < 32; ++w) {
            const int v = w >> 1;
            rank_value(w & 1, v, prev[w & 1][v], 32u * (ntiles - 1u) + 8u * (v / 4) + 4u * h + v % 4 < nl);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        uint64_t bits[F];
#pragma unroll
        for (int s = 0; s < F; ++s) bits[s] = (uint64_t)__double_as_longlong(best[r][s]);
        write_best<F>(p, bits, row0 + 32u * r, lane);
    }
}

template <int KS, int F>
int launch_kf(const D0AssignParams &p, dim3 grid, hipStream_t stream) {
    constexpr int lds = 2 * D0Tile<KS>::kBytes;
    if (ensure_lds_limit(reinterpret_cast<const void *>(&d0_assign_kernel<KS, F>), (int)lds)) return -1;
    hipLaunchKernelGGL((d0_assign_kernel<KS, F>), grid, dim3(kThreads), lds, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int KS, int F>
int launch_wide(const D0AssignParams &p, dim3 grid, hipStream_t stream) {
    constexpr int lds = D0WideTile<KS>::kBytes;
    if (ensure_lds_limit(reinterpret_cast<const void *>(&d0_assign_wide_kernel<KS, F>), (int)lds)) return -1;
    hipLaunchKernelGGL((d0_assign_wide_kernel<KS, F>), grid, dim3(kWideThreads), lds, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int KS>
int launch_ks(const D0AssignParams &p, hipStream_t stream) {
    const uint64_t blocks = (p.rows + kWaves * 32 - 1) / (kWaves * 32);
    if (blocks > 0x7fffffffull) return -2;
    const dim3 grid((uint32_t)blocks);
    // Short lists (the builds replicate to two leaders) are ranked without a
    // branch, so the ranking can stand between the MFMAs: 64 rows per wave.  At
    // 1,000 leaders 1.08-1.3x faster over 5,000 to 400,000 rows and 50 to 1,024
    // columns, at 129 to 480 leaders 1.02-1.6x (30,000 to 2M rows, two or three
    // per row); at 40 leaders up to 4 us slower (one wave per SIMD has the rows'
    // load to itself for only two tiles).  2F - 1 instructions per value make
    // longer lists the slower ones that way.
    const bool wide = p.leaders > kWideLeaders;
    if (p.fanout <= 2) return wide ? launch_wide<KS, 2>(p, grid, stream) : launch_kf<KS, 2>(p, grid, stream);
    if (p.fanout <= 4) return wide ? launch_wide<KS, 4>(p, grid, stream) : launch_kf<KS, 4>(p, grid, stream);
    if (p.fanout <= 8) return launch_kf<KS, 8>(p, grid, stream);
    if (p.fanout <= 16) return launch_kf<KS, 16>(p, grid, stream);
    return launch_kf<KS, 32>(p, grid, stream);
}

// Child histogram with per-workgroup counts in LDS (bins = leaders + 1 words,
// dynamic LDS), added to the global counts once per workgroup and bin: the
// ~1,000 global counters would otherwise take one atomic per fragment.
__global__ __launch_bounds__(256) void d0_hist_lds_kernel(const uint32_t *child, uint64_t n, uint32_t bins,
                                                          uint64_t *counts) {
    extern __shared__ uint32_t hist[];
    for (uint32_t b = threadIdx.x; b < bins; b += blockDim.x) hist[b] = 0u;
    __syncthreads();
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t b = child[i] + 1u;
        if (b < bins) atomicAdd(&hist[b], 1u);
        else atomicAdd(reinterpret_cast<unsigned long long *>(&counts[b]), 1ull);  // not a leader index
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bins; b += blockDim.x)
        if (hist[b]) atomicAdd(reinterpret_cast<unsigned long long *>(&counts[b]), (unsigned long long)hist[b]);
}

__global__ void d0_hist_kernel(const uint32_t *child, uint64_t n, uint64_t *counts) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        atomicAdd(reinterpret_cast<unsigned long long *>(&counts[child[i] + 1]), 1ull);
}

__global__ void d0_fill_zero(uint64_t *a, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = 0ull;
}

// inclusive scan of counts[1..n] in place (one workgroup; n = leaders is small)
__global__ __launch_bounds__(1024) void d0_scan_kernel(uint64_t *counts, uint32_t n) {
    __shared__ uint64_t part[1024];
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint32_t b = 0; b < n; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        part[threadIdx.x] = i < n ? counts[i + 1] : 0ull;
        __syncthreads();
        for (uint32_t off = 1; off < 1024; off <<= 1) {
            const uint64_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0ull;
            __syncthreads();
            part[threadIdx.x] += v;
            __syncthreads();
        }
        if (i < n) counts[i + 1] = carry + part[threadIdx.x];
        __syncthreads();
        if (threadIdx.x == 0) carry += part[1023];
        __syncthreads();
    }
}

uint32_t key_bits(uint32_t leaders) {
    uint32_t b = 1;
    while (b < 32 && (1ull << b) < leaders) ++b;
    return b;
}

}  // namespace

int launch_d0_assign(const D0AssignParams &p, hipStream_t stream) {
    if (p.fanout == 0 || p.fanout > kD0MaxFanout || p.fanout > p.leaders || p.padded_dim % 16 != 0) return -3;
    hipLaunchKernelGGL(d0_rank_kernel, dim3((p.leaders + 255) / 256), dim3(256), 0, stream, p.leader_ids, p.leaders,
                       p.leader_rank, p.rank_leader);
    if (hipGetLastError() != hipSuccess) return -1;
    if (p.rows == 0) return 0;
    const uint32_t ks = (p.padded_dim + 31) / 32;
    if (ks <= 4) return launch_ks<4>(p, stream);
    if (ks <= 8) return launch_ks<8>(p, stream);
    if (ks <= 16) return launch_ks<16>(p, stream);
    if (ks <= 24) return launch_ks<24>(p, stream);
    if (ks <= 32) return launch_ks<32>(p, stream);
    return -3;
}

size_t d0_group_temp_bytes(uint64_t items, uint32_t leaders) {
    size_t sort_bytes = 0;
    hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                       (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)items, 0,
                                       (int)key_bits(leaders));
    // sorted keys, then the sort's own storage (256-byte aligned)
    return ((items * 4 + 255) / 256) * 256 + sort_bytes;
}

int launch_d0_group(const D0AssignParams &p, uint64_t *child_offsets, uint32_t *child_points, void *temp,
                    size_t temp_bytes, hipStream_t stream) {
    const uint64_t items = p.rows * p.fanout;
    hipLaunchKernelGGL(d0_fill_zero, dim3(((uint64_t)p.leaders + 256) / 256), dim3(256), 0, stream, child_offsets,
                       (uint64_t)p.leaders + 1);
    if (items == 0) return hipGetLastError() == hipSuccess ? 0 : -1;
    uint64_t hg = (items + 255) / 256;
    const uint32_t bins = p.leaders + 1u;
    if (bins <= 16384u) {
        hg = hg > 512 ? 512 : hg;
        hipLaunchKernelGGL(d0_hist_lds_kernel, dim3((uint32_t)hg), dim3(256), bins * 4u, stream, p.out_child, items,
                           bins, child_offsets);
    } else {
        hg = hg > 8192 ? 8192 : hg;
        hipLaunchKernelGGL(d0_hist_kernel, dim3((uint32_t)hg), dim3(256), 0, stream, p.out_child, items,
                           child_offsets);
    }
    hipLaunchKernelGGL(d0_scan_kernel, dim3(1), dim3(1024), 0, stream, child_offsets, p.leaders);
    const size_t keys_bytes = ((items * 4 + 255) / 256) * 256;
    uint32_t *keys_out = reinterpret_cast<uint32_t *>(temp);
    size_t sort_bytes = temp_bytes - keys_bytes;
    if (hipcub::DeviceRadixSort::SortPairs(reinterpret_cast<char *>(temp) + keys_bytes, sort_bytes, p.out_child,
                                           keys_out, p.out_point, child_points, (int)items, 0,
                                           (int)key_bits(p.leaders), stream) != hipSuccess)
        return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tessa
