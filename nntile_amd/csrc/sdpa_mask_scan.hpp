// What a workgroup finds out about the rows of a mask given as values before it
// walks the keys, shared by the 16-bit and the fp32 prefill kernels.
#pragma once

#include <type_traits>

#include "sdpa_common.hpp"

namespace nntile_hip
{

// Scan of the mask rows of one query block over the key steps [s_lo, s_hi):
// bit s of not_open: some value of the step s of KEYS keys is not "open", of not_hidden:
// not "hidden" (steps from 63 on share bit 63).  NWAVES wavefronts; words:
// 2 * NWAVES of LDS; the results are the same in every thread.  mask: the
// block's first row; ES: bytes per element; open / hidden: the 32-bit pattern
// of visible / hidden elements.
//
// A lane keeps to one step while it walks the rows, so that what it finds is
// two words ORed and ANDed together (four instructions a load) and a ballot at the end
// says which steps.  Reads of a
// row are contiguous whatever its length; rows and starts that are not
// multiples of 16 bytes only cost some loads a second cache line.  The last
// chunk of a row is moved back to end with the row: it then looks at elements
// of the chunk before once more, which can only make the answer more careful.
// (Before, a lane's loads fell on changing steps, each needing two 64-bit
// shifts, and every lane added its words to LDS with atomics of its own: 7 us
// for the 32 KiB of a 128 x 128 tile, and masks with rows of any other length
// were not scanned at all.)
template<int ES, int NWAVES, int KEYS>
__device__ __forceinline__ void mask_scan_steps(const char *mask, uint32_t ld_bytes, int n_rows,
        int row_bytes, int s_lo, int s_hi, uint32_t open_word, uint32_t hidden_word,
        unsigned long long *words, unsigned long long &not_open_out,
        unsigned long long &not_hidden_out)
{
    constexpr int CPS = KEYS * ES / 16;        // chunks per step
    constexpr int SPAN = 64 / CPS;              // steps that fit a wavefront's lanes
    typedef u32x4 __attribute__((aligned(1))) u32x4_any;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long not_open = 0ull, not_hidden = 0ull;
    // lanes per row: the steps asked for, a power of two, at most all lanes
    int steps_wide = SPAN;
    while(steps_wide > 1 && steps_wide / 2 >= s_hi - s_lo)
    {
        steps_wide >>= 1;
    }
    const int lanes_row = steps_wide * CPS;
    const int rows_pass = (64 / lanes_row) * NWAVES;    // rows one load of everybody covers
    const int r0 = wave * (64 / lanes_row) + lane / lanes_row;
    const int my_step = (lane % lanes_row) / CPS;
    for(int s0 = s_lo; s0 < s_hi; s0 += steps_wide)
    {
        const bool mine = s0 + my_step < s_hi;
        const int at = min((s0 + my_step) * KEYS * ES + (lane % CPS) * 16, row_bytes - 16);
        // (three-operand ors and ands, in two chains)
        uint32_t all_or[2] = {0u, 0u}, all_and[2] = {~0u, ~0u};
        // N loads in flight per lane: eight where they cover the rows (what a small
        // tile's workgroup executes once costs its fetch: 128 x 128 10.8 us with 16
        // and an exclusive or per word, 10.4 so), else 16
        auto look = [&](auto n_tag) __attribute__((always_inline))
        {
            constexpr int N = decltype(n_tag)::value;
            for(int base = 0; base < n_rows; base += N * rows_pass)
            {
                u32x4 v[N];
#pragma unroll
                for(int u = 0; u < N; ++u)
                {
                    // (rows past the end re-read the last one: no branches, so
                    // that the loads are in flight together)
                    const uint32_t row = (uint32_t)min(base + r0 + u * rows_pass, n_rows - 1);
                    v[u] = *reinterpret_cast<const u32x4_any *>(mask + row * ld_bytes + at);
                }
#pragma unroll
                for(int u = 0; u < N; ++u)
                {
                    all_or[0] |= v[u][0] | v[u][1];
                    all_or[1] |= v[u][2] | v[u][3];
                    all_and[0] &= v[u][0] & v[u][1];
                    all_and[1] &= v[u][2] & v[u][3];
                }
            }
        };
        if(n_rows <= 8 * rows_pass)
        {
            look(std::integral_constant<int, 8>{});
        }
        else
        {
            look(std::integral_constant<int, 16>{});
        }
        const uint32_t or_all = all_or[0] | all_or[1], and_all = all_and[0] & all_and[1];
        const uint32_t any_open = (or_all ^ open_word) | (and_all ^ open_word);
        const uint32_t any_hidden = (or_all ^ hidden_word) | (and_all ^ hidden_word);
        const unsigned long long b_open = __builtin_amdgcn_ballot_w64(mine && any_open != 0u);
        const unsigned long long b_hidden = __builtin_amdgcn_ballot_w64(mine && any_hidden != 0u);
        for(int l = 0; l < 64; l += CPS)
        {
            const unsigned long long bit = 1ull << min(s0 + (l % lanes_row) / CPS, 63);
            if(((b_open >> l) & ((1ull << CPS) - 1ull)) != 0ull)
            {
                not_open |= bit;
            }
            if(((b_hidden >> l) & ((1ull << CPS) - 1ull)) != 0ull)
            {
                not_hidden |= bit;
            }
        }
    }
    if(lane == 0)
    {
        words[2 * wave] = not_open;
        words[2 * wave + 1] = not_hidden;
    }
    __syncthreads();
    not_open = not_hidden = 0ull;
#pragma unroll
    for(int w = 0; w < NWAVES; ++w)
    {
        not_open |= words[2 * w];
        not_hidden |= words[2 * w + 1];
    }
    not_open_out = not_open;
    not_hidden_out = not_hidden;
}

} // namespace nntile_hip
