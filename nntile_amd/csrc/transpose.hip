// dst = alpha * src^T for an m x n matrix in Fortran order (element (i, j) of
// src at i + j*m, element (j, i) of dst at j + i*n), the step that moves the
// projections into the attention layout and the attention output back
// (src/kernel/transpose/cpu.cc:21-43 is the arithmetic: one product in fp32,
// one rounding to the tile type).  A workgroup moves a 64 x 64 block through
// LDS: reads run along i, writes along j, both over whole 64-element rows.
#include "sdpa_common.hpp"

namespace nntile_hip
{

struct TrF32
{
    typedef float storage;
    static __device__ __forceinline__ float to_float(float v) { return v; }
    static __device__ __forceinline__ float from_float(float v) { return v; }
};
struct TrBf16
{
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_float(uint16_t v) { return Bf16::to_float(v); }
    static __device__ __forceinline__ uint16_t from_float(float v) { return Bf16::from_float(v); }
};
struct TrFp16
{
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_float(uint16_t v) { return Fp16::to_float(v); }
    static __device__ __forceinline__ uint16_t from_float(float v) { return Fp16::from_float(v); }
};

constexpr int kTrTile = 64;

template<typename S>
__global__ __launch_bounds__(256)
void transpose_kernel(int64_t m, int64_t n, int64_t tiles_m, float alpha,
        const typename S::storage *src, typename S::storage *dst)
{
    typedef typename S::storage E;
    // one column of padding: the transposed reads of a wave fall on 64 banks
    __shared__ E tile[kTrTile][kTrTile + (sizeof(E) == 2 ? 2 : 1)];
    const int64_t i0 = (int64_t)(blockIdx.x % tiles_m) * kTrTile;
    const int64_t j0 = (int64_t)(blockIdx.x / tiles_m) * kTrTile;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    // tile[j][i] = src(i0 + i, j0 + j): 64 consecutive i per wave load
#pragma unroll
    for(int r = 0; r < 16; ++r)
    {
        const int j = ty * 16 + r;
        if(i0 + tx < m && j0 + j < n)
        {
            tile[j][tx] = src[(i0 + tx) + (j0 + j) * m];
        }
    }
    __syncthreads();
    // dst(j0 + j, i0 + i) = alpha * tile[j][i]: 64 consecutive j per wave store
#pragma unroll
    for(int r = 0; r < 16; ++r)
    {
        const int i = ty * 16 + r;
        if(i0 + i < m && j0 + tx < n)
        {
            dst[(j0 + tx) + (i0 + i) * n] = S::from_float(alpha * S::to_float(tile[tx][i]));
        }
    }
}

// 16-bit tiles with m and n multiples of 8 and 16-byte aligned buffers: a
// block of 128 (i) x 32 (j) per workgroup, 16 bytes per global access.  A
// thread reads 8 consecutive i of two neighbouring columns, pairs them into
// 32-bit words (i, j..j+1) and writes those to LDS row i; then it reads 8
// consecutive j of one row and stores them as one 16-byte chunk, a wave 64
// neighbouring chunks.  With n == 32 the block is one contiguous piece of dst.
#ifndef NNTILE_TR16_ITERS
#define NNTILE_TR16_ITERS 1
#endif
constexpr int kTr16Iters = NNTILE_TR16_ITERS;       // 128 rows i per iteration
constexpr int kTr16I = 128 * kTr16Iters, kTr16J = 32, kTr16Pitch = kTr16J / 2 + 1;   // pitch in words

template<typename S>
__global__ __launch_bounds__(256)
void transpose16_kernel(int64_t m, int64_t n, int64_t tiles_m, float alpha,
        const uint16_t *src, uint16_t *dst)
{
    __shared__ uint32_t tile[kTr16I * kTr16Pitch];
    const int64_t i0 = (int64_t)(blockIdx.x % tiles_m) * kTr16I;
    const int64_t j0 = (int64_t)(blockIdx.x / tiles_m) * kTr16J;
    const int tid = threadIdx.x;
    {
        const int c = tid % 16, jp = tid / 16;          // 8 rows i, column pair
        const int64_t j = j0 + 2 * jp;
        u32x4 a[kTr16Iters], b[kTr16Iters];
#pragma unroll
        for(int it = 0; it < kTr16Iters; ++it)
        {
            const int64_t i = i0 + 128 * it + 8 * c;
            a[it] = u32x4{0, 0, 0, 0};
            b[it] = u32x4{0, 0, 0, 0};
            if(i < m && j < n)
            {
                a[it] = __builtin_nontemporal_load(
                        reinterpret_cast<const u32x4 *>(src + i + j * m));
                b[it] = __builtin_nontemporal_load(
                        reinterpret_cast<const u32x4 *>(src + i + (j + 1) * m));
            }
        }
#pragma unroll
        for(int it = 0; it < kTr16Iters; ++it)
        {
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                // a[e] holds rows 2e, 2e+1 of column j; b[e] those of column j+1
                const int r = 128 * it + 8 * c + 2 * e;
                tile[r * kTr16Pitch + jp] = (a[it][e] & 0xffffu) | (b[it][e] << 16);
                tile[(r + 1) * kTr16Pitch + jp] = (a[it][e] >> 16) | (b[it][e] & 0xffff0000u);
            }
        }
    }
    __syncthreads();
    // a wave stores 64 neighbouring 16-byte chunks: 4 chunks (32 columns) a row
#pragma unroll
    for(int q = 0; q < 2 * kTr16Iters; ++q)
    {
        const int k = tid + 256 * q;
        const int r = k / 4, part = k % 4;
        const int64_t i = i0 + r, j = j0 + 8 * part;
        uint32_t w[4];
#pragma unroll
        for(int x = 0; x < 4; ++x)
        {
            w[x] = tile[r * kTr16Pitch + 4 * part + x];
        }
        if(alpha != 1.0f)
        {
#pragma unroll
            for(int x = 0; x < 4; ++x)
            {
                const float lo = alpha * S::to_float((uint16_t)(w[x] & 0xffffu));
                const float hi = alpha * S::to_float((uint16_t)(w[x] >> 16));
                w[x] = (uint32_t)S::from_float(lo) | ((uint32_t)S::from_float(hi) << 16);
            }
        }
        if(i < m && j < n)
        {
            __builtin_nontemporal_store(u32x4{w[0], w[1], w[2], w[3]},
                    reinterpret_cast<u32x4 *>(dst + j + i * n));
        }
    }
}

// Matrices with one short axis of 2 .. 64 (the heads of a layer: projections
// into the attention layout and back).  A block of either kernel above fills
// only as much of its own short side as the matrix has - 8 heads left three
// threads in four idle, 12 heads went element by element - so here a
// workgroup takes kTrShortBytes of the matrix whatever its short axis: `tl`
// long indices, a flat contiguous piece on the side where the short axis is
// the fast one, rows of tl elements on the other.  Both sides move 16 bytes per
// thread; the elements cross over in LDS.
//   SRC_SHORT: src is [long][short]; LDS rows are the short index, padded by 16
//   bytes, and leave as they lie.
//   otherwise: dst is [long][short]; LDS holds the flat piece of dst, with 4
//   bytes of padding behind every 16 bytes x short, so that the lanes of a
//   write, that far apart, fall on different banks.
// Bound: HBM.  bf16, back to back: 8 x 262144 7.9 -> 3.6 us (a launch), 8 x 1163520
// 27.8 -> 7.6 = 4.9 TB/s, 12 x 1163520 53.6 -> 11.3, 32 x 1163520 35.4 -> 26.0 =
// 5.7 TB/s; fp32 16 x 1163520 92.5 -> 26.2.
constexpr int kTrShortMax = 64, kTrShortBytes = 16384;

template<typename S, bool SRC_SHORT>
__global__ __launch_bounds__(256)
void transpose_short_kernel(int n_short, int64_t n_long, int tile_long, float alpha,
        const typename S::storage *src, typename S::storage *dst)
{
    typedef typename S::storage E;
    constexpr int V = 16 / (int)sizeof(E);              // elements per access
    constexpr int ELEMS = kTrShortBytes / (int)sizeof(E);
    constexpr int ITERS = ELEMS / V / 256;
    constexpr int WORD = 4 / (int)sizeof(E);
    __shared__ __attribute__((aligned(16))) E lds[ELEMS
        + (kTrShortMax * V > ELEMS / 8 ? kTrShortMax * V : ELEMS / 8)];
    const int64_t l0 = (int64_t)blockIdx.x * tile_long;
    const int tl = (int)min((int64_t)tile_long, n_long - l0);   // a multiple of V
    const int row_vecs = tl / V, n_vecs = n_short * row_vecs;
    const int pitch = tile_long + V;
    // (quotients by the two wave-common divisors: exact below 2^16)
    const uint32_t by_short = 0xffffffffu / (uint32_t)n_short + 1u;
    const uint32_t by_row = 0xffffffffu / (uint32_t)row_vecs + 1u;
    auto over = [](int x, uint32_t magic, int d) __attribute__((always_inline)) -> int
    {
        return d == 1 ? x : (int)__umulhi((uint32_t)x, magic);
    };
    const int tid = threadIdx.x;
    const E *flat_src = src + l0 * n_short;
    u32x4 raw[ITERS];
#pragma unroll
    for(int it = 0; it < ITERS; ++it)
    {
        const int v = min(tid + 256 * it, n_vecs - 1);
        const int r = over(v, by_row, row_vecs);
        raw[it] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(SRC_SHORT
                    ? flat_src + v * V : src + r * n_long + l0 + (v - r * row_vecs) * V));
    }
#pragma unroll
    for(int it = 0; it < ITERS; ++it)
    {
        const int v = tid + 256 * it;
        if(v >= n_vecs)
        {
            break;
        }
        int at, step, i = 0;
        if(SRC_SHORT)
        {
            const int j = over(v * V, by_short, n_short);
            i = v * V - j * n_short;
            at = i * pitch + j;
            step = pitch;
        }
        else
        {
            const int j = over(v, by_row, row_vecs), c = v - j * row_vecs;
            at = c * (V * n_short + WORD) + j;
            step = n_short;
        }
#pragma unroll
        for(int k = 0; k < V; ++k)
        {
            const uint32_t word = raw[it][k / WORD];
            if constexpr(sizeof(E) == 2)
            {
                lds[at] = (E)(word >> (16 * (k % 2)));
            }
            else
            {
                lds[at] = __uint_as_float(word);
            }
            at += step;
            if(SRC_SHORT && ++i == n_short)
            {
                i = 0;
                at += 1 - n_short * pitch;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for(int it = 0; it < ITERS; ++it)
    {
        const int v = tid + 256 * it;
        if(v >= n_vecs)
        {
            break;
        }
        uint32_t w[4];
        E *to;
        if(SRC_SHORT)
        {
            const int r = over(v, by_row, row_vecs), c = v - r * row_vecs;
            const u32x4 x = *reinterpret_cast<const u32x4 *>(lds + r * pitch + c * V);
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                w[e] = x[e];
            }
            to = dst + r * n_long + l0 + c * V;
        }
        else
        {
            const uint32_t *x = reinterpret_cast<const uint32_t *>(lds + v * V
                    + over(v, by_short, n_short) * WORD);
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                w[e] = x[e];
            }
            to = dst + l0 * n_short + v * V;
        }
        if(alpha != 1.0f)
        {
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                if constexpr(sizeof(E) == 2)
                {
                    const float lo = alpha * S::to_float((uint16_t)(w[e] & 0xffffu));
                    const float hi = alpha * S::to_float((uint16_t)(w[e] >> 16));
                    w[e] = (uint32_t)S::from_float(lo) | ((uint32_t)S::from_float(hi) << 16);
                }
                else
                {
                    w[e] = __float_as_uint(alpha * __uint_as_float(w[e]));
                }
            }
        }
        __builtin_nontemporal_store(u32x4{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4 *>(to));
    }
}

template<typename S>
static int launch_transpose_typed(hipStream_t stream, int64_t m, int64_t n, float alpha,
        const void *src, void *dst)
{
    typedef typename S::storage E;
    const bool aligned = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst))
            & 15u) == 0;
    {
        // a short axis, and a long one of whole 16-byte pieces
        constexpr int V = 16 / (int)sizeof(E);
        const int64_t n_short = m < n ? m : n, n_long = m < n ? n : m;
        if(aligned && n_short >= 2 && n_short <= kTrShortMax && n_long % V == 0 && n_long >= 64)
        {
            const int tile = kTrShortBytes / (int)sizeof(E) / (int)n_short / 32 * 32;
            const int64_t wgs = (n_long + tile - 1) / tile;
            if(wgs > 0x7fffffff)
            {
                return NNTILE_HIP_EINVAL;
            }
            if(m < n)
            {
                hipLaunchKernelGGL((transpose_short_kernel<S, true>), dim3((unsigned)wgs),
                        dim3(256), 0, stream, (int)n_short, n_long, tile, alpha,
                        static_cast<const E *>(src), static_cast<E *>(dst));
            }
            else
            {
                hipLaunchKernelGGL((transpose_short_kernel<S, false>), dim3((unsigned)wgs),
                        dim3(256), 0, stream, (int)n_short, n_long, tile, alpha,
                        static_cast<const E *>(src), static_cast<E *>(dst));
            }
            return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
        }
    }
    if constexpr(sizeof(E) == 2)
    {
        if(m % 8 == 0 && n % 8 == 0 && aligned)
        {
            const int64_t tm = (m + kTr16I - 1) / kTr16I, tn = (n + kTr16J - 1) / kTr16J;
            if(tm > 0x7fffffff / tn)
            {
                return NNTILE_HIP_EINVAL;
            }
            hipLaunchKernelGGL((transpose16_kernel<S>), dim3((unsigned)(tm * tn)), dim3(256), 0,
                    stream, m, n, tm, alpha, static_cast<const uint16_t *>(src),
                    static_cast<uint16_t *>(dst));
            return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
        }
    }
    const int64_t tiles_m = (m + kTrTile - 1) / kTrTile, tiles_n = (n + kTrTile - 1) / kTrTile;
    if(tiles_m > 0x7fffffff / tiles_n)
    {
        return NNTILE_HIP_EINVAL;
    }
    hipLaunchKernelGGL((transpose_kernel<S>), dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0,
            stream, m, n, tiles_m, alpha, static_cast<const E *>(src), static_cast<E *>(dst));
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

// dtype: 0 bf16, 1 fp16, 2 fp32
int launch_transpose(hipStream_t stream, int dtype, int64_t m, int64_t n, float alpha,
        const void *src, void *dst)
{
    switch(dtype)
    {
        case 0: return launch_transpose_typed<TrBf16>(stream, m, n, alpha, src, dst);
        case 1: return launch_transpose_typed<TrFp16>(stream, m, n, alpha, src, dst);
        case 2: return launch_transpose_typed<TrF32>(stream, m, n, alpha, src, dst);
        default: return NNTILE_HIP_EINVAL;
    }
}

} // namespace nntile_hip
