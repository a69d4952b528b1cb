// Rotary position embedding and its backward on a (2, m, n) tensor with
// sines and cosines of shape (m) (src/kernel/rope/cpu.cc:22-52,
// src/kernel/rope_backward/cpu.cc:22-53 are the arithmetic this follows):
//
//   forward:   dst[2i,j]   = cos[i] src[2i,j] - sin[i] src[2i+1,j]
//              dst[2i+1,j] = sin[i] src[2i,j] + cos[i] src[2i+1,j]
//   backward:  dx[2i,j]    = cos[i] dy[2i,j] + sin[i] dy[2i+1,j]
//              dx[2i+1,j]  = cos[i] dy[2i+1,j] - sin[i] dy[2i,j]
//
// (the backward writes dx, it does not add to it).  Products and sums in fp32,
// one rounding to the tile type.  Pure streaming, bound by HBM: a thread takes
// four neighbouring pairs - 16 bytes of a 16-bit tensor, 32 of an fp32 one -
// of COLS columns j and the four sines and cosines that go with them, which it
// so reads once for all of them (read again for every column they are as many
// bytes from L2 as the tensor has); the grid has one axis for i and one for j,
// so that nothing is divided (a 64-bit remainder per thread before).  m not a
// multiple of 4, or addresses that are not aligned for that, take one pair per
// thread.  2 x 131072 x 32 bf16 (34.1 MB) 7.9 -> 6.6 us = 5.2 TB/s; two columns against
// four: 6.6 and 7.1 us there, 14.9 and 15.6 on 2 x 524288 x 8 fp32.
#include "sdpa_common.hpp"

namespace nntile_hip
{

struct RopeF32
{
    typedef float storage;
    static __device__ __forceinline__ float to_float(float v) { return v; }
    static __device__ __forceinline__ float from_float(float v) { return v; }
};
struct RopeBf16
{
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_float(uint16_t v) { return Bf16::to_float(v); }
    static __device__ __forceinline__ uint16_t from_float(float v) { return Bf16::from_float(v); }
};
struct RopeFp16
{
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_float(uint16_t v) { return Fp16::to_float(v); }
    static __device__ __forceinline__ uint16_t from_float(float v) { return Fp16::from_float(v); }
};

template<bool BACKWARD>
__device__ __forceinline__ void rotate(float c, float s, float a, float b, float &x, float &y)
{
    if(BACKWARD)
    {
        x = fmaf(c, a, s * b);
        y = fmaf(c, b, -(s * a));
    }
    else
    {
        x = fmaf(c, a, -(s * b));
        y = fmaf(s, a, c * b);
    }
}

template<typename S, bool BACKWARD, int COLS>
__global__ __launch_bounds__(256)
void rope_vec_kernel(int64_t m, int n, int row_blocks, const typename S::storage *sin,
        const typename S::storage *cos, const typename S::storage *src,
        typename S::storage *dst)
{
    typedef typename S::storage E;
    constexpr int NV = (int)sizeof(E) / 2;      // 16-byte pieces of four pairs
    const int j0 = (int)(blockIdx.x / (unsigned)row_blocks) * COLS;
    const int64_t i = 4 * ((int64_t)(blockIdx.x % (unsigned)row_blocks) * 256 + threadIdx.x);
    if(i >= m)
    {
        return;
    }
    __attribute__((aligned(16))) E sv[4];
    __attribute__((aligned(16))) E cv[4];
    // src and dst pass through once (non-temporal); sin and cos are re-read
    // by the other columns and stay cached
    if constexpr(sizeof(E) == 2)
    {
        *reinterpret_cast<u32x2 *>(sv) = *reinterpret_cast<const u32x2 *>(sin + i);
        *reinterpret_cast<u32x2 *>(cv) = *reinterpret_cast<const u32x2 *>(cos + i);
    }
    else
    {
        *reinterpret_cast<u32x4 *>(sv) = *reinterpret_cast<const u32x4 *>(sin + i);
        *reinterpret_cast<u32x4 *>(cv) = *reinterpret_cast<const u32x4 *>(cos + i);
    }
    u32x4 raw[COLS][NV];
#pragma unroll
    for(int c = 0; c < COLS; ++c)
    {
        // (columns past the end re-read the last one)
        const E *from = src + 2 * (i + m * min(j0 + c, n - 1));
#pragma unroll
        for(int v = 0; v < NV; ++v)
        {
            raw[c][v] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(from) + v);
        }
    }
#pragma unroll
    for(int c = 0; c < COLS; ++c)
    {
        __attribute__((aligned(16))) E in[8];
        __attribute__((aligned(16))) E out[8];
#pragma unroll
        for(int v = 0; v < NV; ++v)
        {
            reinterpret_cast<u32x4 *>(in)[v] = raw[c][v];
        }
#pragma unroll
        for(int k = 0; k < 4; ++k)
        {
            float x, y;
            rotate<BACKWARD>(S::to_float(cv[k]), S::to_float(sv[k]), S::to_float(in[2 * k]),
                    S::to_float(in[2 * k + 1]), x, y);
            out[2 * k] = S::from_float(x);
            out[2 * k + 1] = S::from_float(y);
        }
        if(j0 + c < n)
        {
            E *to = dst + 2 * (i + m * (j0 + c));
#pragma unroll
            for(int v = 0; v < NV; ++v)
            {
                __builtin_nontemporal_store(reinterpret_cast<const u32x4 *>(out)[v],
                        reinterpret_cast<u32x4 *>(to) + v);
            }
        }
    }
}

template<typename S, bool BACKWARD>
__global__ __launch_bounds__(256)
void rope_pair_kernel(int64_t m, int64_t pairs, const typename S::storage *sin,
        const typename S::storage *cos, const typename S::storage *src,
        typename S::storage *dst)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if(t >= pairs)
    {
        return;
    }
    const int64_t i = t % m;
    float x, y;
    rotate<BACKWARD>(S::to_float(cos[i]), S::to_float(sin[i]), S::to_float(src[2 * t]),
            S::to_float(src[2 * t + 1]), x, y);
    dst[2 * t] = S::from_float(x);
    dst[2 * t + 1] = S::from_float(y);
}

template<typename S, bool BACKWARD>
static int launch_rope_typed(hipStream_t stream, int64_t m, int64_t n, const void *sin_,
        const void *cos_, const void *src_, void *dst_)
{
    typedef typename S::storage E;
    const E *sin = static_cast<const E *>(sin_), *cos = static_cast<const E *>(cos_);
    const E *src = static_cast<const E *>(src_);
    E *dst = static_cast<E *>(dst_);
    const int64_t pairs = m * n;
    auto aligned = [](const void *p, uintptr_t a)
    {
        return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
    };
    const bool vec = m % 4 == 0 && n <= 0x7fffffff && aligned(src, 16) && aligned(dst, 16)
        && aligned(sin, 4 * sizeof(E)) && aligned(cos, 4 * sizeof(E));
    if(vec)
    {
        // two columns a thread once that leaves every CU eight workgroups,
        // enough for its memory pipeline
        constexpr int COLS = 2;
        const int64_t rows = (m / 4 + 255) / 256;
        const bool many = rows * ((n + COLS - 1) / COLS) >= 2048;
        const int64_t cols = many ? (n + COLS - 1) / COLS : n;
        if(rows > 0x7fffffff / cols)
        {
            return NNTILE_HIP_EINVAL;
        }
        const dim3 grid((unsigned)(rows * cols));
        if(many)
        {
            hipLaunchKernelGGL((rope_vec_kernel<S, BACKWARD, COLS>), grid, dim3(256), 0, stream, m,
                    (int)n, (int)rows, sin, cos, src, dst);
        }
        else
        {
            hipLaunchKernelGGL((rope_vec_kernel<S, BACKWARD, 1>), grid, dim3(256), 0, stream, m,
                    (int)n, (int)rows, sin, cos, src, dst);
        }
    }
    else
    {
        const int64_t blocks = (pairs + 255) / 256;
        if(blocks > 0x7fffffff)
        {
            return NNTILE_HIP_EINVAL;
        }
        hipLaunchKernelGGL((rope_pair_kernel<S, BACKWARD>), dim3((unsigned)blocks), dim3(256), 0,
                stream, m, pairs, sin, cos, src, dst);
    }
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

// dtype: 0 bf16, 1 fp16, 2 fp32
int launch_rope(hipStream_t stream, int dtype, bool backward, int64_t m, int64_t n,
        const void *sin, const void *cos, const void *src, void *dst)
{
    switch(dtype * 2 + (backward ? 1 : 0))
    {
        case 0: return launch_rope_typed<RopeBf16, false>(stream, m, n, sin, cos, src, dst);
        case 1: return launch_rope_typed<RopeBf16, true>(stream, m, n, sin, cos, src, dst);
        case 2: return launch_rope_typed<RopeFp16, false>(stream, m, n, sin, cos, src, dst);
        case 3: return launch_rope_typed<RopeFp16, true>(stream, m, n, sin, cos, src, dst);
        case 4: return launch_rope_typed<RopeF32, false>(stream, m, n, sin, cos, src, dst);
        case 5: return launch_rope_typed<RopeF32, true>(stream, m, n, sin, cos, src, dst);
        default: return NNTILE_HIP_EINVAL;
    }
}

} // namespace nntile_hip
