// The key axis of a one-tile forward shared out over workgroups: how many
// ranges a call takes, and the kernel that merges what they leave.
#include "sdpa_common.hpp"

namespace nntile_hip
{

// Chunks of a prompt against a filled cache - more rows than the decode
// kernels take, fewer query blocks than the chip has CUs - leave most CUs
// idle while each workgroup walks the whole key axis.  The keys are shared out
// over the idle ones, in the number of ranges that the measured times say is
// best: a step of a workgroup alone on its CU takes kStep (64 keys x 128
// queries of 16 bits, 32 keys x 32 queries of fp32; a second workgroup on a CU
// gains little, so there are 256 places), writing and merging the ranges 3.5 us
// plus 0.7 us for each 10^6 bytes they leave.  Where that is not 1 us faster the
// keys stay together (32 heads, 400 rows, 1100 keys in two ranges: 21.3 -> 27.3
// us).  32 heads over 8: 17 rows, 16000 keys 160 -> 35 us, 100 rows, 8000 keys
// 86 -> 29; fp32, 12 heads, 100 rows, 4000 keys 96 -> 29.
PrefillParts prefill_parts(bool fp32, int64_t batch, int64_t q_seq, int64_t k_seq, int64_t head)
{
    constexpr int64_t kMost = 32, kPlaces = 256;
    const int64_t rows = fp32 ? 32 : 128, keys = fp32 ? 32 : 64;    // of a workgroup, of a step
    const int64_t groups = fp32 ? 4 : 2;    // sets of wavefronts that take steps in turn
    const double kStep = fp32 ? (head == 64 ? 0.72 : 1.33) : (head == 64 ? 0.46 : 0.6);
    const int64_t n_wg = batch * ((q_seq + rows - 1) / rows);
    const int64_t steps = (k_seq + keys - 1) / keys;
    const double part_bytes = 4.0 * (double)batch * (double)q_seq * (double)(head + 2);
    PrefillParts best = {1, 0, 0};
    if(head != 64 && head != 128)
    {
        return best;
    }
    double least = kStep * (double)steps - 1.0;
    for(int64_t want = 2; want <= kMost && want * n_wg <= kPlaces; ++want)
    {
        // (whole rounds of the groups)
        const int64_t each = ((steps + want - 1) / want + groups - 1) / groups * groups;
        const int64_t n = (steps + each - 1) / each;
        const double cost = kStep * (double)each + 3.5 + 0.7e-6 * (double)n * part_bytes;
        if(n > 1 && cost < least)
        {
            least = cost;
            best = {(int)n, (int)(each * keys),
                (size_t)n * batch * q_seq * (head + 2) * sizeof(float)};
        }
    }
    return best;
}

template<typename T> struct PartsOut
{
    typedef uint16_t elem;
    static __device__ __forceinline__ f32x4 load(const elem *at)
    {
        const u32x2 raw = *reinterpret_cast<const u32x2 *>(at);
        return f32x4{T::to_float((uint16_t)(raw[0] & 0xffffu)), T::to_float((uint16_t)(raw[0] >> 16)),
            T::to_float((uint16_t)(raw[1] & 0xffffu)), T::to_float((uint16_t)(raw[1] >> 16))};
    }
    static __device__ __forceinline__ void store(elem *at, f32x4 v)
    {
        *reinterpret_cast<u32x2 *>(at) = u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
    }
};
template<> struct PartsOut<float>
{
    typedef float elem;
    static __device__ __forceinline__ f32x4 load(const elem *at)
    {
        return *reinterpret_cast<const f32x4 *>(at);
    }
    static __device__ __forceinline__ void store(elem *at, f32x4 v)
    {
        *reinterpret_cast<f32x4 *>(at) = v;
    }
};

// Merges the ranges of each row and folds the result into (lse, A).  A thread
// handles 4 head values of one row.  Bound by the latency of its loads, so
// eight ranges travel in one round trip.
template<typename T, int HEAD>
__global__ __launch_bounds__(256)
void sdpa_parts_merge_kernel(const PrefillParams p)
{
    constexpr int TPR = HEAD / 4;               // threads per row
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    const int64_t n_rows = (int64_t)p.batch * p.q_seq;
    const int64_t row = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
    if(row >= n_rows)
    {
        return;
    }
    const int d4 = (threadIdx.x % TPR) * 4;
    float top = neg_inf(), l = 0.0f;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for(int s0 = 0; s0 < p.n_parts; s0 += 8)
    {
        f32x2 ml[8];
        f32x4 v[8];
#pragma unroll
        for(int j = 0; j < 8; ++j)
        {
            // (past the last range: that range again, with weight 0)
            const int64_t prow = min(s0 + j, p.n_parts - 1) * n_rows + row;
            ml[j] = *reinterpret_cast<const f32x2 *>(p.part_ml + 2 * prow);
            v[j] = *reinterpret_cast<const f32x4 *>(p.part_o + prow * HEAD + d4);
        }
        float m_new = top;
#pragma unroll
        for(int j = 0; j < 8; ++j)
        {
            m_new = fmaxf(m_new, ml[j][0]);
        }
        if(m_new == neg_inf())
        {
            continue;       // nothing visible so far
        }
        const float keep = top == neg_inf() ? 0.0f : __expf(top - m_new);
        l *= keep;
        acc *= keep;
#pragma unroll
        for(int j = 0; j < 8; ++j)
        {
            if(s0 + j < p.n_parts && ml[j][0] != neg_inf())
            {
                const float w = __expf(ml[j][0] - m_new);
                l += w * ml[j][1];
                acc += w * v[j];
            }
        }
        top = m_new;
    }
    auto *dst = static_cast<typename PartsOut<T>::elem *>(p.A[0]) + row * HEAD + d4;
    // (a row with a NaN among its scores: as the kernels without ranges do it)
    if(l == 0.0f || (!(l > 0.0f) && !p.overwrite))
    {
        // no visible key
        if(p.overwrite)
        {
            PartsOut<T>::store(dst, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
            if(d4 == 0)
            {
                p.lse[0][row] = neg_inf();
            }
        }
        return;
    }
    const float lse_old = p.overwrite ? neg_inf() : p.lse[0][row];
    float w_old, w_new, lse_out;
    merge_weights(lse_old, top + __logf(l), w_old, w_new, lse_out);
    acc *= w_new / l;
    if(w_old != 0.0f)
    {
        acc += w_old * PartsOut<T>::load(dst);
    }
    PartsOut<T>::store(dst, acc);
    // The threads of a row sit in one wavefront (TPR <= 32 divides 64) and run
    // in lock step: all of them have read lse_old by now.
    if(d4 == 0)
    {
        p.lse[0][row] = lse_out;
    }
}

template<typename T>
int launch_parts_merge(hipStream_t stream, const PrefillParams &p, int head)
{
    const int64_t per_wg = 256 / (head / 4);
    const dim3 grid((unsigned)(((int64_t)p.batch * p.q_seq + per_wg - 1) / per_wg));
    if(head == 64)
    {
        hipLaunchKernelGGL((sdpa_parts_merge_kernel<T, 64>), grid, dim3(256), 0, stream, p);
    }
    else
    {
        hipLaunchKernelGGL((sdpa_parts_merge_kernel<T, 128>), grid, dim3(256), 0, stream, p);
    }
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

template int launch_parts_merge<Bf16>(hipStream_t, const PrefillParams &, int);
template int launch_parts_merge<Fp16>(hipStream_t, const PrefillParams &, int);
template int launch_parts_merge<float>(hipStream_t, const PrefillParams &, int);

} // namespace nntile_hip
