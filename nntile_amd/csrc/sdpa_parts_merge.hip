// The key axis of a one-tile forward shared out over workgroups: how many
// ranges a call takes, and the kernel that merges what they leave.
#include "sdpa_common.hpp"

namespace nntile_hip
{

// Chunks of a prompt against a filled cache - more rows than the decode
// kernels take, fewer query blocks than the chip has CUs - leave most CUs
// idle while each workgroup walks the whole key axis.  The keys are shared out
// over the idle ones, in the number of ranges that the measured times say is
// best: a step of a workgroup alone on its CU takes the time given below (a second
// workgroup on a CU gains little, so there are 256 places), writing and merging the
// ranges 3.5 us plus 0.7 us for each 10^6 bytes they leave.  Where that is not 1 us
// faster the keys stay together (32 heads, 400 rows, 1100 keys in two ranges: 21.3
// -> 27.3 us).  32 heads over 8: 17 rows, 16000 keys 160 -> 35 us, 100 rows, 8000
// keys 86 -> 29.
//
// In fp32 there are two kernels to take the ranges.  The one on fp16 pairs has twice
// the rows, so twice the ranges fit, and is through its keys sooner, but is 4 us
// behind from the start (its longer code and the splitting of the first rows).  us,
// ranges with 32 queries of fp32 products / with 64 of fp16 pairs: 12 heads of 64,
// 65 rows, 365 keys 15.2 / 16.3; 100 rows, 600 keys 15.6 / 17.4, 1100 17.2 / 19.1,
// 4000 32.3 / 26.5; 256 rows, 2256 keys 37.6 / 26.1; 32 heads of 128 over 8, 33 rows,
// 933 keys 24.4 / 21.6; 100 rows, 4100 keys 104.5 / 56.5.
PrefillParts prefill_parts(bool fp32, int64_t batch, int64_t q_seq, int64_t k_seq, int64_t head)
{
    constexpr int64_t kMost = 32, kPlaces = 256;
    struct Kernel
    {
        int form;
        int64_t rows, keys;     // of a workgroup, of a step
        int64_t groups;         // sets of wavefronts that take steps in turn
        double step[2];         // us, head 64 and 128
        double later;           // us behind the other from the start
    };
    static const Kernel kernels[] = {{0, 128, 64, 2, {0.46, 0.6}, 0.0},
        {2, 32, 32, 4, {0.72, 1.33}, 0.0}, {10, 64, 64, 1, {1.13, 2.17}, 4.0}};
    PrefillParts best = {1, 0, 0, 0};
    if(head != 64 && head != 128)
    {
        return best;
    }
    const double part_bytes = 4.0 * (double)batch * (double)q_seq * (double)(head + 2);
    const Kernel *first = fp32 ? kernels + 1 : kernels, *end = fp32 ? kernels + 3 : kernels + 1;
    auto steps = [&](const Kernel &f) { return (k_seq + f.keys - 1) / f.keys; };
    auto step_time = [&](const Kernel &f) { return f.step[head == 64 ? 0 : 1]; };
    double least = 0.0;
    for(const Kernel *f = first; f != end; ++f)
    {
        const double together = step_time(*f) * (double)steps(*f) + f->later - 1.0;
        least = f == first || together < least ? together : least;
    }
    for(const Kernel *f = first; f != end; ++f)
    {
        const int64_t n_wg = batch * ((q_seq + f->rows - 1) / f->rows);
        for(int64_t want = 2; want <= kMost && want * n_wg <= kPlaces; ++want)
        {
            // (whole rounds of the groups)
            const int64_t each = ((steps(*f) + want - 1) / want + f->groups - 1) / f->groups * f->groups;
            const int64_t n = (steps(*f) + each - 1) / each;
            const double cost = step_time(*f) * (double)each + f->later + 3.5
                + 0.7e-6 * (double)n * part_bytes;
            if(n > 1 && cost < least)
            {
                least = cost;
                best = {(int)n, (int)(each * f->keys),
                    (size_t)n * batch * q_seq * (head + 2) * sizeof(float), f->form};
            }
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
