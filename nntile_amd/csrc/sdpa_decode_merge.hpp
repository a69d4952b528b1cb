// The merge of key splits inside the decode launch that computed them, shared
// by the 16-bit and the fp32 decode kernels.
#pragma once

#include "sdpa_common.hpp"

namespace nntile_hip
{

// A value no earlier call of this process has used; its low four bits are clear.
unsigned long long next_decode_tag();
// Longest wait of a merge workgroup for a flag, in ticks of the 100 MHz clock.
unsigned long long decode_spin_limit_now();
// 64-bit words of the sync area per unit.
int decode_sync_stride(int n_splits, int rows, int head);
// Key splits per unit of a launch of which the chip holds `places` workgroups
// at once, before the limits that the number of key steps sets.
int decode_splits_by_units(int units, int places);
// Where the number of splits of a unit may fall as its key steps grow: up to
// kDecodeDirectSteps one workgroup takes all, up to kDecodeSingleSteps a split
// takes one step, beyond that at least two.
constexpr int kDecodeDirectSteps = 3, kDecodeSingleSteps = 8;
// Whether the units' shares of the XCDs differ too much for the merge to ride
// in the launch; row_bytes: of K and V together.
bool decode_uneven_units(int units, int64_t k_seq, int64_t row_bytes);

// Loads that are served by the L2 (never by a CU's own cache): what one
// workgroup reads of memory another workgroup of the same launch has written.
template<bool COH>
__device__ __forceinline__ unsigned long long ld64(const void *ptr)
{
    if(COH)
    {
        return __hip_atomic_load(
                const_cast<unsigned long long *>(static_cast<const unsigned long long *>(ptr)),
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return *static_cast<const unsigned long long *>(ptr);
}

// The XCD this wavefront runs on (hardware register XCC_ID, bits 3:0).
__device__ __forceinline__ int xcc_id()
{
    return (int)(__builtin_amdgcn_s_getreg((31 << 11) | 20) & 15u);
}

// Unit and split of a main workgroup; false: a place that no unit fills.
// Workgroups are dealt round-robin to the 8 XCDs.  All key splits of a unit go
// to one XCD, and so do the workgroups that merge its partials: the partials
// then stay within one L2 (cfg4: 50.6 -> 50.0 us per step).  Units that do not
// come in eights are laid out as if they did (units8) where the merge rides in
// the launch; the places left over end at once.
__device__ __forceinline__ bool decode_place(const DecodeParams &p, int &unit, int &split)
{
    if(p.units8 != 0)
    {
        const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
        unit = (j / p.n_splits) * 8 + x;
        split = j % p.n_splits;
        return unit < p.n_batch * p.n_head_kv;
    }
    split = blockIdx.x % p.n_splits;
    unit = blockIdx.x / p.n_splits;        // nb + n_batch*hkv
    return true;
}

// The partial is complete in this XCD's L2 once every wavefront's stores have
// been acknowledged.  Each wavefront waits for its own in front of the barrier:
// the barrier itself waits for no memory operation, it is a bare s_barrier
// within a workgroup.  Behind it one flag per merge workgroup of the unit goes
// up, with the number of this XCD in its low bits.
__device__ __forceinline__ void decode_raise_flags(const DecodeParams &p, int unit, int split)
{
    if(p.fenced)
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const int tid = threadIdx.x;
    if(tid < p.merge_blocks_per_unit)
    {
        __hip_atomic_store(p.sync + (int64_t)unit * p.sync_stride + 1 + tid * p.n_splits + split,
                p.tag | (unsigned long long)xcc_id(), __ATOMIC_RELAXED,
                __HIP_MEMORY_SCOPE_AGENT);
    }
}

// A merge workgroup of the fused form: block `idx` behind the main workgroups.
// It is dispatched when main workgroups have left (the hardware starts the
// workgroups of a launch in index order, and the main ones never wait for
// anything), waits until every split of its unit has raised its flag, merges
// its rows and lowers the flags again.
//
// Placement: the workgroups of one launch go round the 8 XCDs in index order,
// so the main workgroups of a unit and its merge workgroups, whose indices
// are equal modulo 8 by construction, share an XCD and its L2: partials
// written by plain stores are there for plain loads once the writer's stores
// are acknowledged, no cache has to be written back or invalidated.  Where
// the round starts is not the launch's to say (XCD 0 on a fresh queue, another
// one after a graph launch or on a second stream - but one start per launch,
// also with several queues dispatching at once), so nothing here assumes a
// particular XCD: every main workgroup puts the number of the XCD it ran on
// (hardware register XCC_ID) into its flag and the merge workgroup compares
// it with its own.  A difference - never seen - is counted and the rows are
// left alone rather than merged from data that may not have arrived.  With
// p.fenced both sides use device-scope fences instead and placement is not
// looked at (for comparison: the fences write back and invalidate whole L2s).
// merge_row(unit, row, first head value) merges four head values of a row;
// timeouts, misplaced: where waits that gave up and splits found elsewhere count.
template<int HEAD, typename MergeRow>
__device__ __forceinline__ void decode_merge_workgroup(const DecodeParams &p, int idx,
        unsigned int *timeouts, unsigned int *misplaced, MergeRow merge_row)
{
    constexpr int TPR = HEAD / 4;               // threads per row
    constexpr int ROWS_PER_WG = 256 / TPR;
    const int tid = threadIdx.x;
    const int x = idx & 7, j = idx >> 3;
    const int unit = (j / p.merge_blocks_per_unit) * 8 + x;
    const int rb = j % p.merge_blocks_per_unit;
    if(unit >= p.n_batch * p.n_head_kv)
    {
        return;         // a place of the last eight that no unit fills
    }
    unsigned long long *flags = p.sync + (int64_t)unit * p.sync_stride + 1 + rb * p.n_splits;
    int bad = 0;
    if(tid < p.n_splits)
    {
        // (the tag's low four bits are clear: the flag carries the writer's XCD there)
        const unsigned long long t0 = wall_clock64();
        unsigned long long seen;
        while(((seen = ld64<true>(flags + tid)) & ~15ull) != p.tag)
        {
            __builtin_amdgcn_s_sleep(4);
            if(wall_clock64() - t0 > p.spin_limit)
            {
                bad = 1;
                break;
            }
        }
        if(!bad && !p.fenced && (int)(seen & 15ull) != xcc_id())
        {
            bad = 2;
        }
    }
    bad = __syncthreads_or(bad);
    if(bad)
    {
        if(tid == 0)
        {
            atomicAdd((bad & 1) ? timeouts : misplaced, 1u);
        }
        return;
    }
    if(p.fenced)
    {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    const int rr = rb * ROWS_PER_WG + tid / TPR;
    if(rr < p.rows)
    {
        merge_row(unit, rr, (tid % TPR) * 4);
    }
    // every partial of these rows has been read: the flags go down for the
    // next call on this workspace (a replay of a captured graph has this
    // call's tag again)
    __syncthreads();
    if(tid < p.n_splits)
    {
        __hip_atomic_store(flags + tid, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

} // namespace nntile_hip
