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
// bytes from L2 as the tensor has).  Threads are numbered through all columns,
// whatever their length, so that none is left over at a column's end (with
// workgroups that kept to one column, 2 x 64 x 65536 took 18.6 us, so 6.9; 2 x 4 x
// 2^20 217, so 7.3; 2 x 1028 x 16320 33.2, so 23.8), and a thread's column is a
// multiplication and a shift (a 64-bit remainder before).  m not a multiple of
// 4, or addresses that are not aligned for that, take one pair per thread.
// bf16, one and two columns a thread: 2 x 65536 x 64 (33.6 MB) 7.3 and 6.9 us =
// 4.9 TB/s, 2 x 65536 x 256 24.0 and 22.3 = 6.0 TB/s; fp32 2 x 65536 x 256 55.1 and
// 52.6.
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

// Quotients of numbers below 2^31 by a fixed divisor: a multiplication by
// 2^32 (2^shift - by) / by + 1, rounded down, an addition and a shift, exact
// for every such number (Granlund and Montgomery 1994, theorem 4.2 with N = 32).
struct RopeDivide
{
    uint32_t by, factor, shift;
    explicit RopeDivide(uint32_t d) : by(d), factor(0), shift(0)
    {
        while((1ull << shift) < d)
        {
            ++shift;
        }
        factor = (uint32_t)((((1ull << shift) - d) << 32) / d + 1);
    }
    __device__ __forceinline__ uint32_t quotient(uint32_t t) const
    {
        return (__umulhi(t, factor) + t) >> shift;
    }
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
void rope_vec_kernel(int64_t m, int n, RopeDivide per_col, const typename S::storage *sin,
        const typename S::storage *cos, const typename S::storage *src,
        typename S::storage *dst)
{
    typedef typename S::storage E;
    constexpr int NV = (int)sizeof(E) / 2;      // 16-byte pieces of four pairs
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    const uint32_t col = per_col.quotient(t);
    const int j0 = (int)col * COLS;
    const int64_t i = 4 * (int64_t)(t - col * per_col.by);
    if(j0 >= n)
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
    const int64_t per_col = m / 4;
    // (a thread's number fits 31 bits)
    const bool vec = m % 4 == 0 && n <= 0x7fffffff && pairs / 4 <= 0x7fffff00 && aligned(src, 16)
        && aligned(dst, 16) && aligned(sin, 4 * sizeof(E)) && aligned(cos, 4 * sizeof(E));
    if(vec)
    {
        // two columns a thread once that leaves every CU eight workgroups,
        // enough for its memory pipeline, and where a column is whole cache
        // lines, or each is touched by two loads far apart (bf16 2 x 4 x 2^20
        // 7.3 us with one column, 10.2 with two; 2 x 1028 x 16320 23.5 and 24.1;
        // 2 x 64 x 262144 23.5 and 22.1)
        const bool many = (pairs / 4 + 511) / 512 >= 2048 && 2 * m * (int64_t)sizeof(E) % 128 == 0;
        const int64_t threads = per_col * (many ? (n + 1) / 2 : n);
        const dim3 grid((unsigned)((threads + 255) / 256));
        const RopeDivide divide((uint32_t)per_col);
        if(many)
        {
            hipLaunchKernelGGL((rope_vec_kernel<S, BACKWARD, 2>), grid, dim3(256), 0, stream, m,
                    (int)n, divide, sin, cos, src, dst);
        }
        else
        {
            hipLaunchKernelGGL((rope_vec_kernel<S, BACKWARD, 1>), grid, dim3(256), 0, stream, m,
                    (int)n, divide, sin, cos, src, dst);
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
