// prune.hip -- the final RobustPrune pass over a neighbour table, one
// wavefront per point.
//
// Reference (paths relative to shear-core/src/): final_prune_pipnn,
// index/inmem_index/pipnn_builder.rs:287-330 (the pool is the point's current
// neighbours with their distance to it; an empty row stays empty), then
// robust_prune / occlude_list, algorithm/prune/prune.rs:17-214: the pool sorted
// by (distance, id) and cut to max_occlusion; alpha passes 1.0, x1.2, .. while
// <= alpha and the result is short of max_degree; in pool order a candidate
// whose occlusion factor is <= the pass's alpha is taken (factor := f32::MAX,
// added unless it is the point itself) and every later candidate whose factor
// is <= alpha gets max(factor, d_j / d(j, taken)), f32::MAX when that
// distance is 0; with saturate and alpha > 1 the result is then filled from
// the pool in order.
//
// The scan over the pool is sequential by definition; the wave runs it with
// uniform control and spreads each taken candidate's factor updates over the
// lanes (one later candidate per lane, its distance to the taken one summed in
// coordinate order).  Rows of at most 64 neighbours whose vectors fit a wave's
// LDS go through robust_prune_lds_kernel; the others through
// robust_prune_kernel, where pool keys (distance bits << 32 | id) are sorted
// in LDS by a wave bitonic network and the factors and the result list live in
// LDS, sized by the table's row width.
#include "kernel_attr.h"
#include "prune_kernels.h"
#include "tessa_device.h"

namespace tessa {

namespace {

constexpr uint32_t kWaves = 4;
constexpr uint32_t kThreads = kWaves * 64;
constexpr uint64_t kNoKey = ~0ull;

struct PruneLds {
    uint64_t *key;
    float *occ;
    uint32_t *res;
};

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ void wave_sort_lds(uint64_t *key, uint32_t n2, uint32_t lane) {
    for (uint32_t k = 2; k <= n2; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t c = lane; c < n2 / 2; c += 64) {
                const uint32_t i = ((c & ~(j - 1u)) << 1) | (c & (j - 1u));
                const uint32_t l = i + j;
                const bool up = (i & k) == 0;
                const uint64_t a = key[i], b = key[l];
                if (up ? b < a : a < b) {
                    key[i] = b;
                    key[l] = a;
                }
            }
            wave_lds_sync();
        }
    }
}

// Squared L2 in coordinate order (as l2_ordered), eight 16-byte (or sixteen
// single) loads of each row in flight: with a few waves per SIMD a load's
// latency per step took most of the time.
template <bool kVec4>
__device__ __forceinline__ float l2_deep(const float *x, const float *q, uint32_t dim) {
    constexpr uint32_t kStep = kVec4 ? 8u : 16u;
    const uint32_t n = kVec4 ? dim / 4u : dim;
    float s = 0.0f;
    auto step = [&](float a, float b) {
        const float t = __fsub_rn(a, b);
        s = __fadd_rn(s, __fmul_rn(t, t));
    };
    uint32_t i = 0;
    for (; i + kStep <= n; i += kStep) {
        if constexpr (kVec4) {
            float4 a[kStep], b[kStep];
#pragma unroll
            for (uint32_t k = 0; k < kStep; ++k) {
                a[k] = reinterpret_cast<const float4 *>(x)[i + k];
                b[k] = reinterpret_cast<const float4 *>(q)[i + k];
            }
#pragma unroll
            for (uint32_t k = 0; k < kStep; ++k) {
                step(a[k].x, b[k].x);
                step(a[k].y, b[k].y);
                step(a[k].z, b[k].z);
                step(a[k].w, b[k].w);
            }
        } else {
            float a[kStep], b[kStep];
#pragma unroll
            for (uint32_t k = 0; k < kStep; ++k) a[k] = x[i + k], b[k] = q[i + k];
#pragma unroll
            for (uint32_t k = 0; k < kStep; ++k) step(a[k], b[k]);
        }
    }
    for (uint32_t c = kVec4 ? 4u * i : i; c < dim; ++c) step(x[c], q[c]);
    return s;
}

template <bool kVec4>
__global__ __launch_bounds__(kThreads) void robust_prune_kernel(RobustPruneParams p, uint32_t pool) {
    extern __shared__ __attribute__((aligned(16))) unsigned char prune_lds[];  // kWaves x pool x (key, occ, res)
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t v = blockIdx.x * kWaves + wave;
    if (v >= p.num_points) return;  // whole wave
    unsigned char *mine = prune_lds + (size_t)wave * pool * 16u;
    const PruneLds w{reinterpret_cast<uint64_t *>(mine), reinterpret_cast<float *>(mine + pool * 8u),
                     reinterpret_cast<uint32_t *>(mine + pool * 12u)};
    const float *xv = p.data + (uint64_t)v * p.dim;
    const uint32_t cnt = p.counts[v];
    const uint32_t deg = cnt < p.row_stride ? cnt : p.row_stride;
    uint32_t n2 = 1;
    while (n2 < deg) n2 <<= 1;
    uint32_t n = 0;
    for (uint32_t s0 = 0; s0 < n2; s0 += 64) {
        const uint32_t s = s0 + lane;
        const uint32_t id = s < deg ? p.targets[(uint64_t)v * p.row_stride + s] : 0xFFFFFFFFu;
        const bool ok = id < p.num_points;
        uint64_t key = kNoKey;
        if (ok) key = ((uint64_t)__float_as_uint(l2_deep<kVec4>(xv, p.data + (uint64_t)id * p.dim, p.dim)) << 32) | id;
        if (s < n2) w.key[s] = key;
        n += (uint32_t)__popcll(__ballot(ok));
    }
    wave_lds_sync();
    wave_sort_lds(w.key, n2, lane);
    if (n > p.max_occlusion) n = p.max_occlusion;
    for (uint32_t i = lane; i < n; i += 64) w.occ[i] = 0.0f;
    wave_lds_sync();

    uint32_t rl = 0;
    if (n > 0) {
        float cur = 1.0f;
        while (cur <= p.alpha && rl < p.max_degree) {
            for (uint32_t i = 0; i < n; ++i) {
                if (rl >= p.max_degree) break;
                if (w.occ[i] > cur) continue;
                const uint64_t ki = w.key[i];
                const uint32_t idi = (uint32_t)ki;
                wave_lds_sync();
                if (lane == 0) {
                    w.occ[i] = kEmptyDist;  // f32::MAX
                    if (idi != v) w.res[rl] = idi;
                }
                if (idi != v) ++rl;
                const float *xi = p.data + (uint64_t)idi * p.dim;
                for (uint32_t j = i + 1 + lane; j < n; j += 64) {
                    const float oj = w.occ[j];
                    if (oj > p.alpha) continue;
                    const uint64_t kj = w.key[j];
                    const float djk = l2_deep<kVec4>(p.data + (uint64_t)(uint32_t)kj * p.dim, xi, p.dim);
                    float nf;
                    if (djk == 0.0f) {
                        nf = kEmptyDist;
                    } else {
                        const float q = __fdiv_rn(__uint_as_float((uint32_t)(kj >> 32)), djk);
                        nf = oj > q ? oj : q;
                    }
                    w.occ[j] = nf;
                }
                wave_lds_sync();
            }
            cur = __fmul_rn(cur, 1.2f);
        }
        if (p.saturate && p.alpha > 1.0f) {
            for (uint32_t i = 0; i < n && rl < p.max_degree; ++i) {
                const uint32_t idi = (uint32_t)w.key[i];
                bool seen = false;
                for (uint32_t r = lane; r < rl; r += 64) seen = seen || (w.res[r] == idi);
                seen = __ballot(seen) != 0ull || idi == v;
                wave_lds_sync();
                if (!seen) {
                    if (lane == 0) w.res[rl] = idi;
                    ++rl;
                }
                wave_lds_sync();
            }
        }
    }
    wave_lds_sync();
    uint32_t *out = p.out_targets + (uint64_t)v * p.max_degree;
    for (uint32_t r = lane; r < p.max_degree; r += 64) out[r] = r < rl ? w.res[r] : 0xFFFFFFFFu;
    if (lane == 0) p.out_counts[v] = rl;
}

// ---- rows of at most 64 neighbours ------------------------------------------
// Lane r holds candidate r of the sorted pool (key, factor, which staged row)
// and result r.  The vectors of the pool and of the point lie in LDS, brought
// once by LDS-DMA: every taken candidate needs its distance to all later ones,
// and each lane reading its own vector from memory (64 lines per load) bound
// the pass at a taken candidate's 1,600 cycles of address work for 100
// coordinates.  20,000 rows of 64, 100-d, saturated: 1,126 -> 707 us; 200,000 of
// 128-d 13.7 -> 9.0 ms; 50,000 of 50-d 3,238 -> 627 us; 20,000 of 200-d 3,584 ->
// 2,114.
// Row stride dim + 4 floats (an odd one for a width that is no multiple of 4),
// so the lanes read different banks.
constexpr uint32_t kStageBytes = 53 * 1024;  // three waves per CU

__host__ __device__ inline uint32_t stage_stride(uint32_t dim) { return dim % 4u == 0u ? dim + 4u : dim | 1u; }

template <bool kVec4>
__device__ __forceinline__ void prune_point(const RobustPruneParams &p, uint32_t v, float *rows, uint32_t lane,
                                            uint32_t stride) {
    const uint32_t dim = p.dim;
    const uint32_t cnt = p.counts[v];
    const uint32_t deg = cnt < p.row_stride ? cnt : p.row_stride;
    uint32_t id = lane < deg ? p.targets[(uint64_t)v * p.row_stride + lane] : 0xFFFFFFFFu;
    const bool ok = id < p.num_points;
    const uint64_t valid = __ballot(ok);
    using lds_ptr = __attribute__((address_space(3))) void *;
    auto stage = [&](uint32_t row, uint32_t at) {
        const float *src = p.data + (uint64_t)row * dim;
        for (uint32_t t = 0; t < dim; t += kVec4 ? 256u : 64u) {
            if constexpr (kVec4) {
                if (t + 4u * lane < dim)
                    __builtin_amdgcn_global_load_lds(static_cast<const void *>(src + t + 4u * lane),
                                                     (lds_ptr)(rows + at * stride + t), 16, 0, 0);
            } else {
                if (t + lane < dim)
                    __builtin_amdgcn_global_load_lds(static_cast<const void *>(src + t + lane),
                                                     (lds_ptr)(rows + at * stride + t), 4, 0, 0);
            }
        }
    };
    wave_lds_sync();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the point before has been read
    for (uint64_t m = valid; m; m &= m - 1ull) {
        const uint32_t j = (uint32_t)__builtin_ctzll(m);
        stage((uint32_t)__builtin_amdgcn_readlane((int)id, (int)j), j);
    }
    stage(v, 64u);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    wave_lds_sync();
    auto readlane64 = [](uint64_t x, uint32_t l) -> uint64_t {
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), (int)l) << 32) |
               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, (int)l);
    };
    // the pool in (distance, id) order: every candidate's place by counting
    uint64_t key = kNoKey;
    if (ok) key = ((uint64_t)__float_as_uint(l2_deep<kVec4>(rows + 64u * stride, rows + lane * stride, dim)) << 32) | id;
    uint32_t place = 0;
    for (uint64_t m = valid; m; m &= m - 1ull) {
        const uint32_t j = (uint32_t)__builtin_ctzll(m);
        const uint64_t kj = readlane64(key, j);
        place += kj < key || (kj == key && j < lane) ? 1u : 0u;
    }
    uint32_t n = (uint32_t)__popcll(valid);
    // lanes without a candidate take the places after them
    if (!ok) place = n + (uint32_t)__popcll(~valid & ((1ull << lane) - 1ull));
    const int to = (int)(place * 4u);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)key);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)(uint32_t)(key >> 32));
    const uint32_t at = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)lane);
    id = lo;
    const float dist = __uint_as_float(hi);
    if (n > p.max_occlusion) n = p.max_occlusion;
    const uint64_t pool = n >= 64u ? ~0ull : (1ull << n) - 1ull;
    const float *mine = rows + at * stride;
    float occ = 0.0f;
    uint32_t res = 0, rl = 0;
    if (n > 0u) {
        float cur = 1.0f;
        while (cur <= p.alpha && rl < p.max_degree) {
            uint64_t ahead = pool;  // candidates this pass has not come to
            while (rl < p.max_degree) {
                const uint64_t m = ahead & __ballot(!(occ > cur));
                if (!m) break;
                const uint32_t i = (uint32_t)__builtin_ctzll(m);
                ahead = i == 63u ? 0ull : pool & (~0ull << (i + 1u));
                const uint32_t idi = (uint32_t)__builtin_amdgcn_readlane((int)id, (int)i);
                if (lane == i) occ = kEmptyDist;  // f32::MAX
                if (idi != v) {
                    if (lane == rl) res = idi;
                    ++rl;
                }
                const uint64_t upd = ahead & __ballot(!(occ > p.alpha));
                if (!upd) continue;
                const float *xi = rows + (uint32_t)__builtin_amdgcn_readlane((int)at, (int)i) * stride;
                if ((upd >> lane) & 1ull) {
                    const float djk = l2_deep<kVec4>(mine, xi, dim);
                    if (djk == 0.0f) {
                        occ = kEmptyDist;
                    } else {
                        const float q = __fdiv_rn(dist, djk);
                        occ = occ > q ? occ : q;
                    }
                }
            }
            cur = __fmul_rn(cur, 1.2f);
        }
        if (p.saturate && p.alpha > 1.0f) {
            for (uint32_t i = 0; i < n && rl < p.max_degree; ++i) {
                const uint32_t idi = (uint32_t)__builtin_amdgcn_readlane((int)id, (int)i);
                if (idi == v || __ballot(lane < rl && res == idi)) continue;
                if (lane == rl) res = idi;
                ++rl;
            }
        }
    }
    uint32_t *out = p.out_targets + (uint64_t)v * p.max_degree;
    for (uint32_t r = lane; r < p.max_degree; r += 64) out[r] = r < rl ? res : 0xFFFFFFFFu;
    if (lane == 0) p.out_counts[v] = rl;
}

template <bool kVec4>
__global__ __launch_bounds__(64) void robust_prune_lds_kernel(RobustPruneParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char prune_lds[];
    float *rows = reinterpret_cast<float *>(prune_lds);  // 64 neighbours, then the point
    const uint32_t lane = threadIdx.x, dim = p.dim;
    const uint32_t stride = kVec4 ? dim + 4u : dim | 1u;
    for (uint32_t v = blockIdx.x; v < p.num_points; v += gridDim.x) prune_point<kVec4>(p, v, rows, lane, stride);
}
}  // namespace

int launch_robust_prune(const RobustPruneParams &p, hipStream_t stream) {
    if (p.num_points == 0) return 0;
    const bool vec4 = p.dim % 4 == 0 && reinterpret_cast<uintptr_t>(p.data) % 16 == 0;
    // an unaligned set of a multiple-of-4 width would be staged at a stride that the lanes share banks at
    const bool staged = p.row_stride <= 64u && (vec4 || p.dim % 4u != 0u) &&
                        65ull * stage_stride(p.dim) * 4u <= kStageBytes;
    if (staged) {
        const int bytes = (int)(65u * stage_stride(p.dim) * 4u);
        auto go = [&](auto kernel) -> int {
            if (ensure_lds_limit(reinterpret_cast<const void *>(kernel), bytes)) return -1;
            hipLaunchKernelGGL(kernel, dim3(p.num_points < (1u << 20) ? p.num_points : 1u << 20), dim3(64), bytes, stream, p);
            return hipGetLastError() == hipSuccess ? 0 : -1;
        };
        return vec4 ? go(robust_prune_lds_kernel<true>) : go(robust_prune_lds_kernel<false>);
    }
    uint32_t pool = 64;
    while (pool < p.row_stride) pool <<= 1;  // at most kPruneMaxPool
    const dim3 grid((p.num_points + kWaves - 1) / kWaves), block(kThreads);
    const int bytes = (int)(kWaves * pool * 16u);
    auto go = [&](auto kernel) -> int {
        if (ensure_lds_limit(reinterpret_cast<const void *>(kernel), bytes)) return -1;
        hipLaunchKernelGGL(kernel, grid, block, bytes, stream, p, pool);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    };
    return vec4 ? go(robust_prune_kernel<true>) : go(robust_prune_kernel<false>);
}

}  // namespace tessa
