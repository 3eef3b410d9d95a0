// sq8_quantize.hip -- per-vector symmetric SQ8 quantizer on the GPU.
//
// Restates dco_sq_int8.rs:1431-1467 bit for bit: max|x| and a *sequential*
// f32 sum of squares in dimension order (the reference's own GPU twin,
// compute_backend.rs:17955-18014, tree-reduces the norm and can differ in the
// last bits; this kernel does not), scale = max|x| / max_code (correctly
// rounded division), code = clamp(round_half_away(x / scale)).  Rows with a
// non-finite value are zeroed and reported.
//
// The sums are sequential per row, so one lane owns one row's sum.  Rows of up
// to 8,192 columns go through sq8_quantize_block_kernel (each row read from
// HBM once; see there), wider ones through sq8_quantize_kernel: a workgroup
// takes 256 rows and walks them in 64-column chunks through a padded LDS tile,
// one thread per row, pass 1 for max|x| and the norm, pass 2 reloading each
// chunk for the codes (HBM traffic per row: 2 * 4 * dim read + padded_dim + 8
// written).
#include "kernel_attr.h"
#include "tessa_device.h"

namespace tessa {

namespace {

constexpr int kQRows = 256;              // rows per workgroup, one per thread
constexpr int kQCols = 64;               // columns per chunk
constexpr int kQStride = kQCols + 1;     // floats per LDS row
constexpr int kQCodeWords = kQCols / 4 + 1;  // u32 code words per LDS row

// One chunk of columns [c0, c0 + w) of rows row0.. into the LDS tile.
template <bool kVec4>
__device__ __forceinline__ void load_chunk(const float *x, uint64_t row0, uint32_t nrows, uint32_t dim, uint32_t c0,
                                           uint32_t w, float *tile) {
    const uint32_t t = threadIdx.x;
    if (kVec4 && (w & 3u) == 0u) {
        // 16 lanes per row, 4 floats each: a wave instruction reads 4 rows
        const uint32_t q = t & 15u;
        for (uint32_t r = t >> 4; r < nrows; r += kQRows / 16) {
            if (4u * q < w) {
                const float4 v = *reinterpret_cast<const float4 *>(x + (row0 + r) * dim + c0 + 4u * q);
                float *o = tile + r * kQStride + 4u * q;
                o[0] = v.x;
                o[1] = v.y;
                o[2] = v.z;
                o[3] = v.w;
            }
        }
    } else {
        const uint32_t c = t & 63u;
        for (uint32_t r = t >> 6; r < nrows; r += kQRows / 64)
            if (c < w) tile[r * kQStride + c] = x[(row0 + r) * dim + c0 + c];
    }
}

template <bool kVec4>
__global__ __launch_bounds__(kQRows) void sq8_quantize_kernel(const float *x, uint64_t rows, uint32_t dim,
                                                              uint32_t padded_dim, float max_code, int8_t *codes,
                                                              float *scales, float *norms,
                                                              unsigned long long *bad_row) {
    __shared__ float tile[kQRows * kQStride];
    __shared__ uint32_t ctile[kQRows * kQCodeWords];
    const uint64_t row0 = (uint64_t)blockIdx.x * kQRows;
    const uint32_t nrows = rows - row0 < (uint64_t)kQRows ? (uint32_t)(rows - row0) : (uint32_t)kQRows;
    const uint32_t t = threadIdx.x;
    const bool mine = t < nrows;
    float max_abs = 0.0f;
    float norm = 0.0f;
    bool finite = true;
    // pass 1: max|x| and the sequential sum of squares
    for (uint32_t c0 = 0; c0 < dim; c0 += kQCols) {
        const uint32_t w = dim - c0 < (uint32_t)kQCols ? dim - c0 : (uint32_t)kQCols;
        __syncthreads();  // the previous chunk has been read
        load_chunk<kVec4>(x, row0, nrows, dim, c0, w, tile);
        __syncthreads();
        if (mine) {
            const float *rowp = tile + t * kQStride;
            for (uint32_t c = 0; c < w; ++c) {
                const float v = rowp[c];
                finite &= isfinite(v);
                max_abs = fmaxf(max_abs, fabsf(v));
                norm = __fadd_rn(norm, __fmul_rn(v, v));
            }
        }
    }
    // zero codes for a non-finite row (reported) or an all-zero row
    const bool zero = !finite || max_abs == 0.0f;
    const float scale = zero ? 1.0f : __fdiv_rn(max_abs, max_code);
    if (mine) {
        scales[row0 + t] = scale;
        norms[row0 + t] = finite ? norm : 0.0f;
        if (!finite && bad_row) atomicMin(bad_row, (unsigned long long)(row0 + t));
    }
    // pass 2: codes, chunk by chunk, through the code tile
    for (uint32_t c0 = 0; c0 < padded_dim; c0 += kQCols) {
        const uint32_t w_in = dim > c0 ? (dim - c0 < (uint32_t)kQCols ? dim - c0 : (uint32_t)kQCols) : 0u;
        const uint32_t w_out = padded_dim - c0 < (uint32_t)kQCols ? padded_dim - c0 : (uint32_t)kQCols;
        __syncthreads();  // the previous chunk's tiles have been read
        if (w_in) load_chunk<kVec4>(x, row0, nrows, dim, c0, w_in, tile);
        __syncthreads();
        if (mine) {
            const float *rowp = tile + t * kQStride;
            for (uint32_t c = 0; c < w_out; c += 4) {
                uint32_t word = 0u;
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e) {
                    int8_t code = 0;
                    if (!zero && c + e < w_in) {
                        float qv = roundf(__fdiv_rn(rowp[c + e], scale));
                        qv = fminf(fmaxf(qv, -max_code), max_code);
                        code = (int8_t)(int)qv;
                    }
                    word |= (uint32_t)(uint8_t)code << (8u * e);
                }
                ctile[t * kQCodeWords + c / 4] = word;
            }
        }
        __syncthreads();
        // rows of codes: w_out / 4 words each, consecutive lanes on consecutive words
        const uint32_t words = w_out / 4u;
        for (uint32_t e = t; e < nrows * words; e += kQRows) {
            const uint32_t r = e / words, qw = e - r * words;
            *reinterpret_cast<uint32_t *>(codes + (row0 + r) * padded_dim + c0 + 4u * qw) = ctile[r * kQCodeWords + qw];
        }
    }
}

// ---- one workgroup per block of rows, the block read once ---------------------
// Rows of up to kBlockMaxDim columns.  A workgroup (four waves) copies its R
// rows to LDS with LDS-DMA loads (global_load_lds: no VGPR round trip), then
// works from LDS only:
//  * wave 0 forms the sums of squares, lane r row r's, in dimension order;
//  * the other waves form max|x| (as an integer maximum of the magnitudes'
//    bits, which also finds a non-finite value) and the codes, 2^k lanes per
//    row, one word of four codes per lane and step, held in registers between
//    the two when a lane has at most kQuads of them.
// The two need nothing from each other.  The sums are a chain of 2 * dim
// dependent instructions for however many lanes have a row, so they bound a
// workgroup of few rows: one wave per 4 rows, sums, maxima and codes in turn,
// took 1.23 ms for 1,048,576 x 768 (3.3 TB/s), this split takes 0.73 ms (5.5
// TB/s); at a width that is no multiple of 4 one thread per row, rows read
// twice and a division per element, 400,003 x 50 took 267 us, now 60 (39 in the
// kernel).  R is the
// largest power of two up to 32 whose rows fit kBlockLds, several workgroups
// per CU (16 rows of 768 in 49 KB: 0.93 ms; 4 of 960: 320 us, 8: 293; 64 of
// 128: 260 us, 32: 212), and that leave 1,024 blocks (with few rows a block's
// own time counts: 920 x 256, the whole call, 38 us with 32 rows, 31 with 4).
// kPad (dim % 4 == 0, 16-byte aligned rows): row stride dim + 4 floats, so the
// row lanes read disjoint banks.  Otherwise the rows lie as they do in memory,
// where the block is one run of floats; a stride that is no multiple of 4
// spreads the row lanes over the banks by itself.
// Codes: q = x * (1/scale) lies within 3 * 2^-24 * |x/scale| < 2.3e-5 of the
// correctly rounded quotient fl(x/scale) (|x/scale| <= max_code < 128), so
// round-half-away of q and of fl(x/scale) agree unless a half-integer lies
// within that distance of q; words with such an element
// (|frac(q) - 0.5| <= 4e-5), and rows whose scale is not a normal float with a
// finite reciprocal, take the correctly rounded division instead.  Codes
// equal the per-element division's bit for bit.
constexpr uint32_t kBlockMaxDim = 8192;        // 128 KB of LDS per block of 4 rows
constexpr uint32_t kBlockLds = 34 * 1024;
constexpr uint32_t kBlockThreads = 256;
constexpr float kHalfMargin = 4.0e-5f;

__device__ __forceinline__ uint32_t exact_code(float v, float scale, float max_code) {
    return (uint32_t)(uint8_t)(int8_t)(int)fminf(fmaxf(roundf(__fdiv_rn(v, scale)), -max_code), max_code);
}

// Four codes as one word.  Fast: no element lies within the margin of a
// half-integer, so round-half-away is round-to-nearest-even, which adding
// 1.5 * 2^23 does (|q| <= 127.0001; the low byte of the sum is the integer).
__device__ __forceinline__ uint32_t quant_word(const float (&v)[4], float inv, float scale, bool fast, float max_code) {
    float q[4], m = 1.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        q[e] = __fmul_rn(v[e], inv);
        m = fminf(m, fabsf(__fsub_rn(__builtin_amdgcn_fractf(q[e]), 0.5f)));
    }
    if (fast && m > kHalfMargin) {
        uint32_t b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = __float_as_uint(__fadd_rn(q[e], 12582912.0f));
        // low bytes of b[0..3]
        return __builtin_amdgcn_perm(__builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u),
                                     __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u), 0x05040100u);
    }
    return exact_code(v[0], scale, max_code) | (exact_code(v[1], scale, max_code) << 8) |
           (exact_code(v[2], scale, max_code) << 16) | (exact_code(v[3], scale, max_code) << 24);
}

template <bool kPad>
__device__ __forceinline__ void read_quad(const float *row, uint32_t c, uint32_t dim, float (&v)[4]) {
    if (kPad) {
        const float4 x = c < dim ? *reinterpret_cast<const float4 *>(row + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) v[e] = c + e < dim ? row[c + e] : 0.0f;
    }
}

__device__ __forceinline__ void dma_floats(const float *src, float *dst, uint32_t n, uint32_t lane, bool vec4) {
    // n floats by one wave; the LDS address of a lane follows from the first lane's
    using lds_ptr = __attribute__((address_space(3))) void *;
    uint32_t at = 0;
    if (vec4)
        for (; at < (n & ~3u); at += 256u)
            if (at + 4u * lane < (n & ~3u))
                __builtin_amdgcn_global_load_lds(static_cast<const void *>(src + at + 4u * lane), (lds_ptr)(dst + at), 16,
                                                 0, 0);
    for (at = vec4 ? n & ~3u : 0u; at < n; at += 64u)
        if (at + lane < n)
            __builtin_amdgcn_global_load_lds(static_cast<const void *>(src + at + lane), (lds_ptr)(dst + at), 4, 0, 0);
}

// lanes: lanes per row of the code waves (a power of two <= 64)
template <bool kPad, int kQuads>
__global__ __launch_bounds__(kBlockThreads) void sq8_quantize_block_kernel(
    const float *x, uint64_t rows, uint32_t dim, uint32_t padded_dim, uint32_t block_rows, uint32_t lanes, bool vec4,
    float max_code, int8_t *codes, float *scales, float *norms, unsigned long long *bad_row) {
    extern __shared__ __attribute__((aligned(16))) float blk[];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint64_t row0 = (uint64_t)blockIdx.x * block_rows;
    const uint32_t nrows = rows - row0 < (uint64_t)block_rows ? (uint32_t)(rows - row0) : block_rows;
    const uint32_t stride = kPad ? dim + 4u : dim;
    if (kPad) {
        for (uint32_t r = wave; r < nrows; r += kBlockThreads / 64u)
            dma_floats(x + (row0 + r) * dim, blk + r * stride, dim, lane, true);
    } else {
        // the run cut into four pieces of a multiple of 4 floats
        const uint32_t n = nrows * dim, piece = ((n / 4u) + 3u) & ~3u;
        const uint32_t a = wave * piece < n ? wave * piece : n;
        const uint32_t b = wave == 3u || a + piece > n ? n : a + piece;
        dma_floats(x + row0 * dim + a, blk + a, b - a, lane, vec4);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    if (wave == 0u) {
        if (lane >= nrows) return;
        const float *row = blk + lane * stride;
        float norm = 0.0f;
        if (kPad) {
            const float4 *row4 = reinterpret_cast<const float4 *>(row);
#pragma unroll 4
            for (uint32_t t = 0; t < dim / 4u; ++t) {
                const float4 v = row4[t];
                norm = __fadd_rn(norm, __fmul_rn(v.x, v.x));
                norm = __fadd_rn(norm, __fmul_rn(v.y, v.y));
                norm = __fadd_rn(norm, __fmul_rn(v.z, v.z));
                norm = __fadd_rn(norm, __fmul_rn(v.w, v.w));
            }
        } else {
#pragma unroll 8
            for (uint32_t t = 0; t < dim; ++t) norm = __fadd_rn(norm, __fmul_rn(row[t], row[t]));
        }
        // a non-finite value makes the sum non-finite; a non-finite sum of
        // finite values (overflow) is told apart by looking at the values
        bool finite = true;
        if (!isfinite(norm))
            for (uint32_t c = 0; c < dim; ++c) finite &= isfinite(row[c]);
        norms[row0 + lane] = finite ? norm : 0.0f;
        return;
    }

    const uint32_t words = padded_dim / 4u;
    const uint32_t per = 64u / lanes;  // rows of a wave at a time
    const uint32_t li = lane & (lanes - 1u);
    for (uint32_t r0 = (wave - 1u) * per; r0 < nrows; r0 += 3u * per) {
        const uint32_t r = r0 + lane / lanes;
        const bool live = r < nrows;
        const float *row = blk + (live ? r : r0) * stride;
        float v[kQuads > 0 ? kQuads : 1][4];
        uint32_t top = 0;
        auto fold = [&](const float (&x4)[4]) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t m = __float_as_uint(x4[e]) & 0x7fffffffu;
                top = top > m ? top : m;
            }
        };
        if constexpr (kQuads > 0) {
#pragma unroll
            for (int k = 0; k < kQuads; ++k) {
                read_quad<kPad>(row, 4u * (li + (uint32_t)k * lanes), dim, v[k]);
                fold(v[k]);
            }
        } else {
            for (uint32_t q = li; q < words; q += lanes) {
                read_quad<kPad>(row, 4u * q, dim, v[0]);
                fold(v[0]);
            }
        }
        for (uint32_t off = lanes / 2u; off > 0u; off >>= 1) {
            const uint32_t o = __shfl_xor(top, (int)off);
            top = top > o ? top : o;
        }
        // zero codes for a non-finite row (reported) or an all-zero row
        const bool finite = top < 0x7f800000u, zero = !finite || top == 0u;
        const float scale = zero ? 1.0f : __fdiv_rn(__uint_as_float(top), max_code);
        const float inv = __fdiv_rn(1.0f, scale);
        const bool fast = scale >= 1.17549435e-38f && isfinite(inv);
        if (live && li == 0u) {
            scales[row0 + r] = scale;
            if (!finite && bad_row) atomicMin(bad_row, (unsigned long long)(row0 + r));
        }
        uint32_t *out = reinterpret_cast<uint32_t *>(codes + (row0 + (live ? r : r0)) * padded_dim);
        if constexpr (kQuads > 0) {
#pragma unroll
            for (int k = 0; k < kQuads; ++k) {
                const uint32_t q = li + (uint32_t)k * lanes;
                const uint32_t word = zero ? 0u : quant_word(v[k], inv, scale, fast, max_code);
                if (live && q < words) out[q] = word;
            }
        } else {
            for (uint32_t q = li; q < words; q += lanes) {
                read_quad<kPad>(row, 4u * q, dim, v[0]);
                const uint32_t word = zero ? 0u : quant_word(v[0], inv, scale, fast, max_code);
                if (live) out[q] = word;
            }
        }
    }
}

template <bool kPad>
int launch_block(const float *x, uint64_t rows, uint32_t dim, uint32_t padded_dim, bool vec4, float max_code,
                 int8_t *codes, float *scales, float *norms, unsigned long long *bad_row, hipStream_t stream) {
    const uint32_t row_bytes = (dim + (kPad ? 4u : 0u)) * 4u;
    uint32_t r = 32;
    while (r > 4u && (r * row_bytes > kBlockLds || rows < 1024ull * r)) r /= 2u;
    const uint64_t nblk = (rows + r - 1) / r;
    if (nblk > 0x7fffffffull) return -2;
    const uint32_t words = padded_dim / 4u;
    uint32_t lanes = 4;
    while (lanes < 64u && lanes < words) lanes *= 2u;
    const uint32_t quads = (words + lanes - 1u) / lanes;
    const int lds = (int)(r * row_bytes);
    auto go = [&](auto kernel) -> int {
        if (ensure_lds_limit(reinterpret_cast<const void *>(kernel), lds)) return -1;
        hipLaunchKernelGGL(kernel, dim3((uint32_t)nblk), dim3(kBlockThreads), lds, stream, x, rows, dim, padded_dim, r,
                           lanes, vec4, max_code, codes, scales, norms, bad_row);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    };
    switch (quads) {
        case 1: return go(sq8_quantize_block_kernel<kPad, 1>);
        case 2: return go(sq8_quantize_block_kernel<kPad, 2>);
        case 3: return go(sq8_quantize_block_kernel<kPad, 3>);
        case 4: return go(sq8_quantize_block_kernel<kPad, 4>);
        default: return go(sq8_quantize_block_kernel<kPad, 0>);
    }
}

__global__ void init_bad_row(unsigned long long *bad_row) { *bad_row = ~0ull; }

}  // namespace

int launch_sq8_quantize(const float *x, uint64_t rows, uint32_t dim, uint32_t padded_dim, uint32_t bits,
                        int8_t *codes, float *scales, float *norms, uint64_t *bad_row, hipStream_t stream) {
    const float max_code = (float)((1u << (bits - 1)) - 1u);
    unsigned long long *bad = (unsigned long long *)bad_row;
    if (bad_row) hipLaunchKernelGGL(init_bad_row, dim3(1), dim3(1), 0, stream, bad);
    if (rows == 0) return 0;
    const bool aligned = (reinterpret_cast<uintptr_t>(x) & 15u) == 0u;
    if (dim <= kBlockMaxDim) {
        // whole words of codes: padded_dim and the code rows are multiples of 4
        if (dim % 4u == 0u && aligned)
            return launch_block<true>(x, rows, dim, padded_dim, true, max_code, codes, scales, norms, bad, stream);
        return launch_block<false>(x, rows, dim, padded_dim, aligned, max_code, codes, scales, norms, bad, stream);
    }
    const uint64_t blocks = (rows + kQRows - 1) / kQRows;
    if (blocks > 0x7fffffffull) return -2;
    if (dim % 4u == 0u && aligned)
        hipLaunchKernelGGL(sq8_quantize_kernel<true>, dim3((uint32_t)blocks), dim3(kQRows), 0, stream, x, rows, dim,
                           padded_dim, max_code, codes, scales, norms, (unsigned long long *)bad_row);
    else
        hipLaunchKernelGGL(sq8_quantize_kernel<false>, dim3((uint32_t)blocks), dim3(kQRows), 0, stream, x, rows,
                           dim, padded_dim, max_code, codes, scales, norms, (unsigned long long *)bad_row);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tessa
