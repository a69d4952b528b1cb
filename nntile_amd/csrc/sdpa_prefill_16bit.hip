// Prefill attention forward for 16-bit tiles (bf16 / fp16) on gfx950.
//
// One workgroup = 4 wavefronts = 128 queries of one (batch entry, query tile);
// each wavefront owns 32 queries.  Keys are walked in steps of 64.
//
//   S^T = K Q^T    v_mfma_f32_32x32x16: A = 32 keys x 16 head values read from
//                  LDS, B = 16 head values x 32 queries held in registers for
//                  the whole kernel.  In the 32x32 accumulator layout a lane
//                  holds ONE query (lane % 32) and 16 of the 32 keys, so the
//                  row maximum and the row sum of the softmax are reductions
//                  over the lane's own registers plus one exchange with lane^32.
//   O^T += V^T P^T A = 32 head values x 16 keys read from LDS, B = P^T taken
//                  straight from the S^T accumulators (converted to 16 bit) -
//                  the accumulator layout of the first product IS the B layout
//                  of the second, up to a fixed permutation of the 16 keys,
//                  and the V operand is gathered in that permuted key order.
//
// K and V steps go from global memory straight into LDS (global_load_lds,
// 16 bytes per lane, no register round trip), double-buffered, one barrier per
// step; the loads of step g+1 are issued at the top of step g.  A load
// instruction fills 1 KB of LDS contiguously, so rows cannot be padded; bank
// conflicts are avoided by XOR-swizzling the 16-byte chunks of a row instead
// (each lane picks the global chunk that belongs at its LDS position).
// V arrives with the head axis contiguous but the second product contracts
// over keys: its MFMA operand is read with ds_read_b64_tr_b16, which hands
// each lane 4 keys of one head value from a 4 x 16 block.
//
// The running (max, sum) pair lives in registers across all key tiles of a
// query tile; the epilogue merges the result into the (lse, A) pair in memory
// (the hand-off between NNTile tasks), so one launch can stand for one task or
// for a whole row of tasks.
#include <algorithm>
#include <atomic>
#include <random>
#include <type_traits>

#include "sdpa_mask_scan.hpp"
#include "sdpa_mask_words.hpp"

#ifndef NNTILE_PF_AHEAD
#define NNTILE_PF_AHEAD 3
#endif

namespace nntile_hip
{

constexpr int kQRows = 128;     // queries per workgroup of four wavefronts
constexpr int kKeys = 64;       // keys per step
constexpr int kThreads = 256;
constexpr unsigned kCUsPerXCD = 32;   // MI355X: 256 CUs in 8 XCDs

// Walks the key steps of all key tiles in order: tile kt, step kb within the
// tile, rows left in the tile from this step on.
struct StepCursor
{
    int kt, kb, rows_left;
    const char *Kp, *Vp;    // first row of the step in the current key tile
};

// ds_read_b64_tr_b16: within each block of 16 lanes, lane i supplies the
// address of 4 consecutive 16-bit values of row i/4 (values 4*(i%4)..+3 of
// 16) and receives value i of rows 0..3.
__device__ __forceinline__ u32x2 lds_read_tr16(const char *lds_ptr)
{
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(lds_ptr));
    return __builtin_bit_cast(u32x2, v);
}

// Developer build (-DNNTILE_PF_TRACE): wall-clock stamps (100 MHz) of every
// workgroup of the last launch - start, first step in LDS, end of the
// pipelined loop, end of the key steps, end - plus where it ran and how many
// steps it had; read back with nntile_hip_debug_pf_trace.
#ifdef NNTILE_PF_TRACE
__device__ unsigned long long pf_trace[8 * 4096];
#define PF_STAMP(i) do { if(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) == 0 \
        && blockIdx.x < 4096) { pf_trace[8 * blockIdx.x + (i)] = wall_clock64(); } } while(0)
#define PF_NOTE(i, v) do { if(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) == 0 \
        && blockIdx.x < 4096) { pf_trace[8 * blockIdx.x + (i)] = (unsigned long long)(v); } } while(0)
extern "C" int nntile_hip_debug_pf_trace(unsigned long long *host)
{
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(pf_trace), sizeof(pf_trace));
}
#else
#define PF_STAMP(i)
#define PF_NOTE(i, v)
#endif

// WAVES: wavefronts per workgroup, 32 queries each.  4: two workgroups share a
// CU.  8 (analytic masks, head 64 and 128): one workgroup of 256 queries per
// CU, whose eight wavefronts share every K/V step - a CU then brings each step
// into LDS once where two workgroups of four bring it twice.
// The scan that is done once for all batch entries: blocks of as many rows as the
// attention workgroups have, each in key ranges, so that a scanning workgroup reads as
// much of blocks of 64 rows (four ranges) as of 128.
template<int ROWS>
constexpr int kScanSplits = ROWS < kQRows ? kMaskBitSplits * ROWS / kQRows : kMaskBitSplits;

// Key range sp of kScanSplits<ROWS> of query block qb.
template<int ES, int NWAVES, int ROWS>
__device__ __forceinline__ void mask_scan_range(const char *mask, uint32_t ld_bytes, int q_len,
        int k_seq, uint32_t open_word, uint32_t hidden_word, int qb, int sp,
        unsigned long long *words, unsigned long long &not_open, unsigned long long &not_hidden)
{
    const int n_steps = (k_seq + kKeys - 1) / kKeys;
    const int per_split = (n_steps + kScanSplits<ROWS> - 1) / kScanSplits<ROWS>;
    const int s_lo = min(sp * per_split, n_steps);
    mask_scan_steps<ES, NWAVES, kKeys>(mask + (int64_t)(qb * ROWS) * ld_bytes, ld_bytes,
            min(ROWS, q_len - qb * ROWS), k_seq * ES, s_lo, min(s_lo + per_split, n_steps),
            open_word, hidden_word, words, not_open, not_hidden);
}

// What a scan found about one (block, key range), as the words of its entry, by one
// thread each.
__device__ __forceinline__ void mask_words_publish(unsigned long long *entry, int tid,
        unsigned long long not_open, unsigned long long not_hidden, unsigned long long tag)
{
    static_assert(MaskWords::N == kMaskBitWords, "an entry holds its words");
    if(tid < kMaskBitWords)
    {
        __hip_atomic_store(entry + tid,
                (unsigned long long)MaskWords::word(tid, tag, not_open, not_hidden),
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Exclusive or of the values of every eight lanes that follow each other
__device__ __forceinline__ uint64_t sum_of_eight(uint64_t x)
{
    uint32_t v[2] = {(uint32_t)x, (uint32_t)(x >> 32)};
#pragma unroll
    for(int w = 0; w < 2; ++w)
    {
        // the neighbour's, the other pair's, the other four's (lanes in reverse)
        v[w] ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[w], 0xb1, 0xf, 0xf, true);
        v[w] ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[w], 0x4e, 0xf, 0xf, true);
        v[w] ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[w], 0x141, 0xf, 0xf, true);
    }
    return ((uint64_t)v[1] << 32) | v[0];
}

// PARTS: the workgroup takes one of p.n_parts ranges of the keys and leaves
// its triple in memory (PrefillParams::part_o), where launch_parts_merge finds it.
// KH == 2: the workgroup's four wavefronts hold 64 queries, and every step's 64 keys
// are shared by two wavefronts of the same 32 queries, 32 keys each; the two
// (maximum, sum, output) triples are merged through LDS before the epilogue.
template<typename T, int HEAD, int MODE, int WAVES = 4, int GROUPS = 1, bool PARTS = false,
    int KH = 1>
__global__ __launch_bounds__(WAVES * 64, WAVES == 4 ? 2 : 1)
void sdpa_prefill_16bit_kernel(const PrefillParams p)
{
    PF_STAMP(0);
    // GROUPS == 2: the eight wavefronts are two groups of four; both groups
    // hold the same 128 queries, group g takes the key steps g, g + 2, ...
    // through a K/V ring of its own, and the two (maximum, sum, output)
    // triples are merged through LDS before the epilogue.  For launches that
    // have no second workgroup to put on a CU: two wavefronts per SIMD (one's
    // softmax beside the other's MFMAs) and half the chain of dependent steps.
    constexpr int QW = WAVES / GROUPS;      // wavefronts that share a key step
    constexpr int ROWS = QW / KH * 32;      // queries of the workgroup
    constexpr int THREADS = WAVES * 64;
    constexpr int SCAN_SPLITS = kScanSplits<ROWS>;
    constexpr int NB = 2 / KH;              // 32-key blocks of a step that a wavefront takes
    typedef typename T::vec8 vec8;
    constexpr int KSTEPS = HEAD / 16;       // MFMA steps along head for S
    constexpr int DBLOCKS = HEAD / 32;      // 32-row blocks of O^T
    constexpr int RB = HEAD * 2;            // bytes per K/V row
    constexpr int CPR = HEAD / 8;           // 16-byte chunks per row
    constexpr int RPL = 16 / CPR;           // rows per 256-byte line of LDS banks
    constexpr int ROWS_PER_LOAD = 1024 / RB;   // rows one load instruction fills
    constexpr int LOADS = kKeys / ROWS_PER_LOAD;  // load instructions per K (or V) step
    constexpr int LOADS_PER_WAVE = LOADS / QW;
    constexpr int K_BYTES = kKeys * RB;
    constexpr int NDB = DBLOCKS / KH;       // blocks of O^T a wavefront writes
    constexpr int RBE = RB / KH;            // bytes of a row it writes
    constexpr int CPRE = CPR / KH;
    constexpr bool EXPLICIT = (MODE == NNTILE_HIP_MASK_ADDITIVE
            || MODE == NNTILE_HIP_MASK_BOOL);
    static_assert(LOADS_PER_WAVE * QW == LOADS
            && (LOADS_PER_WAVE == 1 || LOADS_PER_WAVE == 2 || LOADS_PER_WAVE == 4),
            "head size does not fit this tiling");
    static_assert(GROUPS == 1 || (GROUPS == 2 && WAVES == 8), "two groups of four wavefronts");
    static_assert(!PARTS || (GROUPS == 2 && !EXPLICIT), "parts: analytic masks, two groups");
    static_assert(WAVES == 4 || (WAVES == 8 && (GROUPS == 2 || !EXPLICIT)),
            "eight wavefronts on 256 queries: analytic masks only");
    static_assert(KH == 1 || (KH == 2 && WAVES == 4 && GROUPS == 1 && !PARTS && DBLOCKS % 2 == 0),
            "halved steps: one group of four wavefronts, each left with half of the head");

    // Separate arrays, not one: the compiler then knows that the loads
    // streaming into one of them cannot alias the reads of the others and
    // does not make those reads wait for the loads.  Key step g lives in
    // lds_k[g % 2] and lds_v[g % 2].
    // (GROUPS == 2: group g's half of every array starts at g * K_BYTES; that
    // offset is part of the lanes' read addresses and of the loads' targets)
    __shared__ __attribute__((aligned(1024))) char lds_k0[K_BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_k1[K_BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_v0[K_BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_v1[K_BYTES * GROUPS];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int grp = GROUPS > 1 ? (tid >> 6) / QW : 0;      // which key steps
    const int wave = (tid >> 6) - grp * QW;                 // which 32 queries
    const int lds_grp_off = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(grp) * K_BYTES : 0;
    const int kh = KH > 1 ? __builtin_amdgcn_readfirstlane(wave >> 1) : 0;  // which 32 keys of a step
    const int rb = KH > 1 ? wave & 1 : wave;                // which 32 of its group's queries
    const int col = lane & 31;      // query within the wavefront / row of a block
    const int half = lane >> 5;

    // ---- which queries --------------------------------------------------
    // Workgroups are dealt round-robin to the 8 XCDs.  With xcd_remap every
    // XCD gets a contiguous range of batch entries (their query blocks share
    // K and V in that XCD's L2); in both layouts the query blocks are handed
    // out last-first, all batch entries of a block before the next block, so
    // that under a causal mask the longest workgroups start first.
    //
    // An XCD places its workgroups i = 0..31 on its 32 CUs and i = 32..63
    // beside them, i+32 next to i.  With the plain longest-first order the CU
    // that gets the longest workgroup also gets the longest of the second
    // group, and the CUs end the first round with very different amounts of
    // work done.  The second group is therefore dealt in reverse: the longest
    // workgroup shares its CU with the shortest of the first 64.
    const int q_blocks = p.n_q_tiles * p.q_blocks_per_tile;
    unsigned wg = blockIdx.x, n_att = gridDim.x;     // n_att: attention workgroups
    if constexpr(EXPLICIT)
    {
        // The first workgroups of the grid scan the mask for everybody (one
        // query tile, one key tile): they wait for nothing, so the attention
        // workgroups behind them can wait for their words.
        if(p.n_scan_wgs > 0)
        {
            if((int)blockIdx.x < p.n_scan_wgs)
            {
                constexpr int ES = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 2 : 1;
                __shared__ unsigned long long pub_words[2 * WAVES];
                unsigned long long pub_open, pub_hidden;
                const int scan_blk = (int)blockIdx.x / SCAN_SPLITS;
                if(scan_blk * ROWS >= (int)p.q_seq)
                {
                    return;     // (there to make their number a multiple of 8)
                }
                mask_scan_range<ES, WAVES, ROWS>(static_cast<const char *>(p.mask),
                        (uint32_t)(p.mask_ld * ES), (int)p.q_seq, (int)p.k_seq,
                        (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 0u : 0x01010101u,
                        (MODE == NNTILE_HIP_MASK_ADDITIVE) ? T::kNegInfPair : 0u,
                        scan_blk, (int)blockIdx.x % SCAN_SPLITS, pub_words, pub_open, pub_hidden);
                // written through to memory (device scope), where readers on any
                // XCD find them; the tag says which are there, none waits for another
                mask_words_publish(p.mask_bits + kMaskBitWords * (int64_t)blockIdx.x, tid, pub_open,
                        pub_hidden, p.mask_tag);
                return;
            }
            wg -= (unsigned)p.n_scan_wgs;
            n_att -= (unsigned)p.n_scan_wgs;
        }
    }
    // (as far as it goes: the places it is dealt to must all be attention workgroups' -
    // those that scan a mask do not count.  257 to 511 workgroups of 128 queries, causal,
    // head 128, dealt in order / in reverse: 12 x 4096 71.2 / 67.7 us, 6 x 8192 131 / 124, 20 x 3000
    // 59.2 / 56.5; a window given as values, 64 x 700, 20.8 / 22.6, so those only where the
    // second group is complete)
    if constexpr(WAVES == 4)
    {
        const unsigned i = wg >> 3, n = min(n_att >> 3, 2u * kCUsPerXCD);
        if(i >= kCUsPerXCD && i < n && (KH > 1 || !EXPLICIT || n == 2u * kCUsPerXCD))
        {
            wg = ((kCUsPerXCD + n - 1u - i) << 3) | (wg & 7u);
        }
    }
    // (the parts of a query block have equal indices modulo 8 - one XCD - where
    // the batch entries come in eights)
    int part = 0;
    if constexpr(PARTS)
    {
        const unsigned per_part = gridDim.x / (unsigned)p.n_parts;
        part = (int)(wg / per_part);
        wg -= (unsigned)part * per_part;
    }
    const int part_k0 = PARTS ? part * p.part_keys : 0;
    // (functions, here and below, so that kernels without ranges read their
    // arguments where they use them, as if this were not there)
    auto overwrite = [&]() __attribute__((always_inline)) { return PARTS || p.overwrite; };
    int b, qblk;
    // this workgroup among those of its entry on its XCD
    int my_place = 0, n_places = 0;
    const int batch_all = p.batch * p.n_slabs;
    if(p.xcd_remap)
    {
        const int b_per_xcd = batch_all >> 3;
        const int i = (int)(wg >> 3);
        b = (int)(wg & 7) * b_per_xcd + i % b_per_xcd;
        qblk = q_blocks - 1 - i / b_per_xcd;
        my_place = i / b_per_xcd;
        n_places = q_blocks;
    }
    else if constexpr(KH > 1)
    {
        // Every XCD gets a run of the (entry, query block) pairs, so that it has few
        // entries' keys in its L2.  An entry's blocks lie in the run as longest,
        // shortest, second longest, ...: any piece of an entry is as much work as any
        // other; of a run, the longer ones (even places) come first, then the others
        // from long to short.
        const int x = (int)(wg & 7), i = (int)(wg >> 3);
        const int n = (int)n_att;
        const int run0 = x * (n >> 3) + min(x, n & 7);
        const int run = (n >> 3) + (x < (n & 7) ? 1 : 0), longer = (run + 1) >> 1;
        const int at = run0 + (i < longer ? 2 * i : 2 * (run - 1 - i) + 1);
        b = at / q_blocks;
        const int place = at - b * q_blocks;
        qblk = (place & 1) ? place >> 1 : q_blocks - 1 - (place >> 1);
        const int first_place = max(run0 - b * q_blocks, 0);
        my_place = place - first_place;
        n_places = min(run0 + run - b * q_blocks, q_blocks) - first_place;
    }
    else
    {
        b = (int)wg % batch_all;
        qblk = q_blocks - 1 - (int)wg / batch_all;
    }
    // the slab of this entry: its tiles are allocations of their own
    int q_tile0 = 0, k_tile0 = 0;
    if(p.n_slabs > 1)
    {
        const int slab = b / p.batch;
        b -= slab * p.batch;
        q_tile0 = slab * p.n_q_tiles;
        k_tile0 = slab * p.n_kv_tiles;
    }
    const int qt = qblk / p.q_blocks_per_tile;
    const int qb = qblk % p.q_blocks_per_tile;
    const int q_len = (int)min(p.q_tile, p.q_seq - (int64_t)qt * p.q_tile);
    const int q_row0 = qb * ROWS;                     // within the tile
    if(q_row0 >= q_len)
    {
        return;
    }
    const int kvb = kv_entry(b, p.n_batch, p.kv_group);

    const uint16_t *Qt = static_cast<const uint16_t *>(p.Q[q_tile0 + qt])
        + (int64_t)b * q_len * HEAD;
    const int my_q = q_row0 + rb * 32 + col;            // row within tile
    const bool q_ok = my_q < q_len;
    // the stored logsumexp that the epilogue merges with: requested here, so
    // that its latency passes beside the first loads
    float *lse_ptr = p.lse[q_tile0 + qt] + (int64_t)b * q_len + (q_ok ? my_q : 0);
    const float lse_stored = overwrite() ? neg_inf() : *lse_ptr;

    // Q fragments, resident for the whole kernel.
    vec8 qf[KSTEPS];
    {
        const uint16_t *src = Qt + (int64_t)(q_ok ? my_q : 0) * HEAD + half * 8;
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            u32x4 raw = *reinterpret_cast<const u32x4 *>(src + ks * 16);
            if(!q_ok)
            {
                raw = u32x4{0, 0, 0, 0};
            }
            qf[ks] = __builtin_bit_cast(vec8, raw);
        }
    }

    // ---- which keys --------------------------------------------------------
    // rel0: position of the workgroup's first query minus the position of key
    // row 0, plus the causal offset; key row kg is visible to query row
    // (q_row0 + r) iff kg <= rel0 + r.  Clamped so that the 32-bit arithmetic
    // below cannot overflow.
    const int k_seq = PARTS ? min(p.part_keys, (int)p.k_seq - part_k0) : (int)p.k_seq;
    const int k_tile = PARTS ? k_seq : (int)p.k_tile;
    int rel0 = 0;
    const int last_k_len = k_seq - (p.n_kv_tiles - 1) * k_tile;
    int n_steps = (p.n_kv_tiles - 1) * p.k_blocks_per_tile
        + (last_k_len + kKeys - 1) / kKeys;
    if(MODE == NNTILE_HIP_MASK_CAUSAL)
    {
        int64_t rel = p.q_pos0 + (int64_t)qt * p.q_tile + q_row0
            + p.causal_offset - p.k_pos0 - part_k0;
        rel = max((int64_t)-(1 << 30), min(rel, (int64_t)(1 << 30)));
        rel0 = (int)rel;
        const int hi = min(rel0 + min(ROWS, q_len - q_row0) - 1, k_seq - 1);
        if(hi < 0)
        {
            if(!overwrite())
            {
                return;
            }
            n_steps = 0;    // nothing visible: the epilogue writes empty rows
        }
        else
        {
            const int kt_hi = hi / k_tile;
            n_steps = min(n_steps, kt_hi * p.k_blocks_per_tile
                    + (hi - kt_hi * k_tile) / kKeys + 1);
        }
    }
    const int wave_rel_lo = rel0 + rb * 32;         // first query of the wavefront
    const int my_rel = wave_rel_lo + col;

    // ---- LDS layout and the lane's fixed addresses ---------------------------
    // A step's K (and V) block is kKeys rows of RB bytes, unpadded.  The
    // 16-byte chunk c of row r is stored at chunk position
    //   K:  c ^ ((r / RPL) % CPR)        16 consecutive rows, same c -> 16 bank groups
    //   V:  c ^ (4 * ((r / RPL) % (CPR/4)))   4 consecutive rows x 64 B -> 4 quarters
    // Load instruction `ld` fills rows [ld*ROWS_PER_LOAD, +ROWS_PER_LOAD): lane
    // L lands on row ld*ROWS_PER_LOAD + L/CPR, chunk position L%CPR, and so must
    // fetch the logical chunk that belongs there.
    // (V: the swizzle repeats from one load instruction to the next, so its
    // offsets are v_goff0 + i*1024 and go into the instructions' immediates,
    // which advance the global and the LDS address alike)
    uint32_t k_goff[LOADS_PER_WAVE], v_goff0 = 0;
    int ld_row0 = 0;
    const int ld_cpos = lane % CPR;
#pragma unroll
    for(int i = 0; i < LOADS_PER_WAVE; ++i)
    {
        const int ld = wave * LOADS_PER_WAVE + i;
        const int r = ld * ROWS_PER_LOAD + lane / CPR;
        k_goff[i] = (uint32_t)(r * RB + (ld_cpos ^ ((r / RPL) % CPR)) * 16);
        if(i == 0)
        {
            ld_row0 = r;
            v_goff0 = (uint32_t)(r * RB
                    + (ld_cpos ^ (4 * ((r / RPL) % (CPR >= 4 ? CPR / 4 : 1)))) * 16);
        }
    }
    // S operand: lane (col, half) reads row mb*32+col, logical chunk 2*ks+half.
    // (KH == 2: its one block is block kh of the step, and 32 rows change no swizzle)
    uint32_t k_raddr[NB][KSTEPS];
#pragma unroll
    for(int mb = 0; mb < NB; ++mb)
    {
        const int r = (mb + kh) * 32 + col;
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            k_raddr[mb][ks] = (uint32_t)(grp * K_BYTES + r * RB
                    + ((2 * ks + half) ^ ((r / RPL) % CPR)) * 16);
        }
    }
    // PV operand through the transposing read: within a 16-lane block, lane i
    // addresses key j = i/4 and head values 4*(i%4)..+3 of the block's 16 head
    // values, and receives keys 0..3 of head value i.  Blocks: lanes 16..31
    // take the upper 16 head values of a 32-row block, lanes 32..63 the keys
    // 4..7 (lane half h).  For step t (16 keys) and instruction a (keys
    // 8a + 4h + j) the row is 16t + 8a + 4h + j; 16t + 8a goes into the
    // instruction's immediate offset.
    uint32_t v_raddr[DBLOCKS];
    {
        const int i16 = lane & 15, dblk = (lane >> 4) & 1;
        const int j = i16 >> 2, r4 = i16 & 3;
        const int r = 4 * half + j;         // row modulo 8: enough for the swizzle
        const int swz = 4 * ((r / RPL) % (CPR >= 4 ? CPR / 4 : 1));
#pragma unroll
        for(int db = 0; db < DBLOCKS; ++db)
        {
            // (KH == 2: a wavefront's blocks start with the half of the head that
            // it is left with after the merge)
            const int c = 4 * ((db + kh * (DBLOCKS / 2)) % DBLOCKS) + 2 * dblk + (r4 >> 1);
            v_raddr[db] = (uint32_t)(grp * K_BYTES + (kh * 32 + r) * RB + (c ^ swz) * 16
                    + 8 * (r4 & 1));
        }
    }

    auto tile_rows = [&](int kt) -> int
    {
        return min(k_tile, k_seq - kt * k_tile);
    };

    // Byte offset of batch entry kvb's slab inside key tile kt.
    auto slab = [&](int kt) -> int64_t
    {
        const int64_t rows = p.kv_rows > 0 ? p.kv_rows : (int64_t)tile_rows(kt);
        return (int64_t)kvb * rows * HEAD * 2 + (int64_t)part_k0 * (HEAD * 2);
    };

    // Global -> LDS loads of the K (or V) rows of one step.  Rows past the end
    // of the tile are clamped to its last row: their scores are masked and
    // their probabilities are exactly 0, so any finite stand-in value works.
    auto fetch_k = [&](const StepCursor &cur, char *dst_base)
    {
        // (wave index made visibly uniform: the LDS target goes into M0)
        char *dst = dst_base + lds_grp_off
            + __builtin_amdgcn_readfirstlane(wave) * LOADS_PER_WAVE * 1024;
        if(cur.rows_left >= kKeys)
        {
#pragma unroll
            for(int i = 0; i < LOADS_PER_WAVE; ++i)
            {
                load_to_lds16<0, false>(cur.Kp + k_goff[i], dst + i * 1024);
            }
        }
        else
        {
            const int last = cur.rows_left - 1;
#pragma unroll
            for(int i = 0; i < LOADS_PER_WAVE; ++i)
            {
                // same chunk, clamped row
                const uint32_t back = (uint32_t)(
                        max(ld_row0 + i * ROWS_PER_LOAD - last, 0) * RB);
                load_to_lds16<0, false>(cur.Kp + (k_goff[i] - back), dst + i * 1024);
            }
        }
    };
    auto fetch_v = [&](const StepCursor &cur, char *dst_base)
    {
        char *dst = dst_base + lds_grp_off
            + __builtin_amdgcn_readfirstlane(wave) * LOADS_PER_WAVE * 1024;
        if(cur.rows_left >= kKeys)
        {
            const char *src = cur.Vp + v_goff0;
            load_to_lds16<0, false>(src, dst);
            if(LOADS_PER_WAVE > 1)
            {
                load_to_lds16<1024, false>(src, dst);
            }
            if(LOADS_PER_WAVE > 2)
            {
                load_to_lds16<2048, false>(src, dst);
                load_to_lds16<3072, false>(src, dst);
            }
        }
        else
        {
            const int last = cur.rows_left - 1;
#pragma unroll
            for(int i = 0; i < LOADS_PER_WAVE; ++i)
            {
                const uint32_t back = (uint32_t)(
                        max(ld_row0 + i * ROWS_PER_LOAD - last, 0) * RB);
                load_to_lds16<0, false>(cur.Vp + (v_goff0 + i * 1024 - back), dst + i * 1024);
            }
        }
    };

    // Next step; the tile base pointers are re-read only when the tile changes.
    auto advance_one = [&](StepCursor &cur)
    {
        cur.kb += 1;
        cur.rows_left -= kKeys;
        cur.Kp += kKeys * RB;
        cur.Vp += kKeys * RB;
        if(cur.rows_left <= 0)
        {
            cur.kt += 1;
            cur.kb = 0;
            if(cur.kt < p.n_kv_tiles)
            {
                cur.rows_left = tile_rows(cur.kt);
                cur.Kp = static_cast<const char *>(p.K[k_tile0 + cur.kt]) + slab(cur.kt);
                cur.Vp = static_cast<const char *>(p.V[k_tile0 + cur.kt]) + slab(cur.kt);
            }
            else
            {
                cur.rows_left = 0;
            }
        }
    };
    // ... the next step of this wavefront's group
    auto advance = [&](StepCursor &cur)
    {
        advance_one(cur);
        if(GROUPS > 1)
        {
            advance_one(cur);
        }
    };

    // Score units: the raw dot product is kept and the scale is folded into
    // the exponent; an additive mask value is divided by the scale before it
    // is added, which is the same thing.
    const float c = p.scale * kLog2e;
    const float inv_scale = 1.0f / p.scale;

    // ---- explicit mask tiles ----------------------------------------------------
    // The wavefront's 32 x 64 mask values of a key step are loaded one step ahead
    // as whole pieces of rows: load i brings rows 16*(i%2) + lane/4 and keys
    // 32*(i/2) + 8*(lane%4) .. +7, 16 bytes a lane (boolean: 8).  At the top of the
    // step the wavefront classifies its block from the raw bits: nothing hidden
    // (the step runs as if there were no mask), everything hidden (the step is
    // skipped), or mixed.  Mixed values go through LDS, 32 keys at a time, to the
    // lanes that apply them: lane (col, half) has query my_q and keys
    // mb*32 + 8*rg + 4*half + 0..3.  (Loaded from there directly - eight loads whose
    // lanes lie in 32 rows each - a step took 1.0 to 1.3 us longer: the
    // address path takes a lane a clock when neighbours share no line.  1024 x 1024
    // x 32 of head 128: a window of 65 keys 20.7 -> 16.9 us, causal 26.3 -> 24.4,
    // every step mixed 53.5 -> 38.9.)
    // The loads carry the alignment of one element; in a ragged last step a piece
    // that would reach past the row is moved back to end with it and shifted into
    // place when it is used, and what lies past the end is made hidden.
    constexpr int MW = ((MODE == NNTILE_HIP_MASK_ADDITIVE) ? 16 : 8) / KH;     // dwords per lane and step
    enum { MASK_ZERO = 0, MASK_HIDDEN = 1, MASK_MIXED = 2 };
    uint32_t mraw[MW];
#pragma unroll
    for(int i = 0; i < MW; ++i)
    {
        mraw[i] = 0;
    }
    constexpr int PW = MW / (2 * NB);           // dwords of a piece of eight elements
    constexpr int MASK_RB = 32 * 8 * PW / 16;   // bytes of 32 elements
    constexpr int MASK_RPL = 256 / MASK_RB;     // such rows per 256-byte line of LDS banks
    const int piece = lane & 3, piece_row = lane >> 2;
    // first key of load i's piece within the step, as loaded and as meant
    auto piece_key0 = [&](int i) -> int
    {
        return ((i >> 1) + kh) * 32 + 8 * piece;
    };
    auto piece_start = [&](int key0, int keys) -> int
    {
        // (a row of less than a piece is loaded from its start)
        return max(min(key0, keys - 8), keys == k_seq ? 0 : -kKeys);
    };
    // loads of the mask values of key step kb (of `keys` keys) into mraw
    auto mask_fetch = [&](int kb, int keys)
    {
        typedef typename std::conditional<MODE == NNTILE_HIP_MASK_ADDITIVE, uint16_t,
                uint8_t>::type M;
        typedef typename std::conditional<MODE == NNTILE_HIP_MASK_ADDITIVE, u32x4, u32x2>::type V;
        typedef V __attribute__((aligned(1))) V_any;
        const M *mp[2];
#pragma unroll
        for(int h = 0; h < 2; ++h)
        {
            // (rows past the end of the tile re-read its last one)
            const int row = min(q_row0 + rb * 32 + 16 * h + piece_row, q_len - 1);
            mp[h] = static_cast<const M *>(p.mask) + (int64_t)row * p.mask_ld + kb * kKeys;
        }
        if(k_seq >= 8)
        {
#pragma unroll
            for(int i = 0; i < 2 * NB; ++i)
            {
                const int at = keys >= kKeys ? piece_key0(i) : piece_start(piece_key0(i), keys);
                const V v = *reinterpret_cast<const V_any *>(mp[i & 1] + at);
#pragma unroll
                for(int w = 0; w < PW; ++w)
                {
                    mraw[PW * i + w] = v[w];
                }
            }
        }
        else
        {
            // (rows of less than one piece)
#pragma unroll
            for(int i = 0; i < 2; ++i)
            {
#pragma unroll
                for(int w = 0; w < PW; ++w)
                {
                    constexpr int EPW = 8 / PW;
                    uint32_t x = 0u;
#pragma unroll
                    for(int e = 0; e < EPW; ++e)
                    {
                        x |= (uint32_t)mp[i][min(EPW * w + e, k_seq - 1)] << (32 / EPW * e);
                    }
                    mraw[PW * i + w] = x;
                }
            }
        }
    };
    // brings the pieces of a ragged step of `keys` keys into place
    auto mask_fix_ragged = [&](int keys)
    {
        constexpr int EB = 32 * PW / 8;         // bits of an element
        constexpr uint32_t HIDDEN = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? T::kNegInfPair : 0u;
#pragma unroll
        for(int i = 0; i < 2 * NB; ++i)
        {
            const int key0 = piece_key0(i);
            const int back = key0 - piece_start(key0, keys);
            const int valid = min(max(keys - key0, 0), 8);
#pragma unroll
            for(int w = 0; w < PW; ++w)
            {
                // dword w of the piece moved down by `back` elements
                const int bit = back * EB + 32 * w;
                uint32_t lo = 0u, hi = 0u;
#pragma unroll
                for(int j = w; j < PW; ++j)
                {
                    lo = (bit >> 5) == j ? mraw[PW * i + j] : lo;
                    hi = (bit >> 5) == j - 1 ? mraw[PW * i + j] : hi;
                }
                const uint32_t x = (uint32_t)((((uint64_t)hi << 32) | lo) >> (bit & 31));
                // (its elements from `valid` on are past the end)
                const int n = min(max(valid * EB - 32 * w, 0), 32);
                const uint32_t keep = n == 32 ? ~0u : (1u << n) - 1u;
                mraw[PW * i + w] = (x & keep) | (HIDDEN & ~keep);
            }
        }
    };
    // hands the pieces to the lanes that apply them: group i (keys (i/4)*32 +
    // 8*(i%4) + 4*half + 0..3 of query my_q) into dwords PW/2 * i .. of mraw.
    // Chunk c of row r sits at chunk position c ^ (r / MASK_RPL) % 4 of its 32 keys:
    // 256 bytes that are read together lie in different banks.
    auto mask_transpose = [&]() __attribute__((always_inline))
    {
        typedef typename std::conditional<MODE == NNTILE_HIP_MASK_ADDITIVE, u32x4, u32x2>::type V;
        __shared__ __attribute__((aligned(16))) char lds_mask[EXPLICIT ? WAVES * 32 * MASK_RB : 16];
        char *mine = lds_mask + (tid >> 6) * (32 * MASK_RB);
#pragma unroll
        for(int mb = 0; mb < NB; ++mb)
        {
#pragma unroll
            for(int h = 0; h < 2; ++h)
            {
                const int r = 16 * h + piece_row;
                V v;
#pragma unroll
                for(int w = 0; w < PW; ++w)
                {
                    v[w] = mraw[PW * (2 * mb + h) + w];
                }
                *reinterpret_cast<V *>(mine + r * MASK_RB
                        + (piece ^ ((r / MASK_RPL) % 4)) * (4 * PW)) = v;
            }
            // (the LDS accesses of a wavefront are carried out in order; this
            // keeps the compiler to it)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for(int rg = 0; rg < 4; ++rg)
            {
                const char *at = mine + col * MASK_RB + (rg ^ ((col / MASK_RPL) % 4)) * (4 * PW)
                    + half * (2 * PW);
                if constexpr(MODE == NNTILE_HIP_MASK_ADDITIVE)
                {
                    const u32x2 v = *reinterpret_cast<const u32x2 *>(at);
                    mraw[2 * (4 * mb + rg)] = v[0];
                    mraw[2 * (4 * mb + rg) + 1] = v[1];
                }
                else
                {
                    mraw[4 * mb + rg] = *reinterpret_cast<const uint32_t *>(at);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    };
    auto mask_classify = [&]() -> int
    {
        uint32_t all_or = 0u, all_and = 0xffffffffu;
#pragma unroll
        for(int i = 0; i < MW; ++i)
        {
            all_or |= mraw[i];
            all_and &= mraw[i];
        }
        bool lane_open, lane_hidden;
        if(MODE == NNTILE_HIP_MASK_ADDITIVE)
        {
            lane_open = (all_or == 0u);                 // every value is +0
            lane_hidden = (all_or == T::kNegInfPair) && (all_and == T::kNegInfPair);
        }
        else
        {
            lane_open = (all_or == 0x01010101u) && (all_and == 0x01010101u);
            lane_hidden = (all_or == 0u);
        }
        if(__builtin_amdgcn_ballot_w64(!lane_open) == 0)
        {
            return MASK_ZERO;
        }
        if(__builtin_amdgcn_ballot_w64(!lane_hidden) == 0)
        {
            return MASK_HIDDEN;
        }
        return MASK_MIXED;
    };

    f32x16 o[DBLOCKS];
#pragma unroll
    for(int db = 0; db < DBLOCKS; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            o[db][r] = 0.0f;
        }
    }
    float m_run = neg_inf();
    float l_run = 0.0f;      // this lane half's share of the row sum

    PHASE_DECL
    StepCursor cur = {0, 0, tile_rows(0),
        static_cast<const char *>(p.K[k_tile0]) + slab(0),
        static_cast<const char *>(p.V[k_tile0]) + slab(0)};     // step being computed
    if(GROUPS > 1 && grp == 1)
    {
        advance_one(cur);       // the second group starts at step 1
    }
    StepCursor nxt = cur;                        // step being fetched
    // Masks given as values: what the loop most likely starts with - the first
    // step's K and V and the K of the step behind it - is requested before the
    // mask is looked at (below: a wait for the scanning workgroups' flags, or a
    // scan of this workgroup's own rows).  What the mask then says may make
    // any of it unnecessary, which costs nothing but the request.  (Not the
    // first step's mask values: 16 loads that touch 32 rows each delay the
    // scan more than they save, 6 % on 4 x 4 tiles of 355 keys.)
    // Workgroups of 64 queries are twice as many, and together their requests delay the
    // scan: those that scan for themselves make none, nor do the others of a
    // launch of about a workgroup a CU and more (two at head 64).  us, every workgroup's
    // requests made / not, what a mask hides wholly: head 128, 32 x 500 4.7 / 4.3, 16 x 2048
    // 8.8 / 7.6; head 64, 32 x 1024 5.0 / 4.5, 24 x 2000 7.3 / 6.9, 64 x 700 5.4 / 4.9; below
    // that the others lose by it: 9 x 1700 of head 128, causal, 26.3 / 27.3, 4 x 2048 open 26.7 /
    // 27.5, 16 x 1024 of head 64 open 15.3 / 15.9, 36 x 500 causal 12.1 / 12.6.  Without a
    // shared scan, hidden: 16 x 1500 of head 128 14.9 / 14.2, 24 x 2000 of head 64 18.8 / 17.9, causal
    // 34.7 / 35.1.
    const bool early = KH == 1 || (p.mask_bits != nullptr && n_att * HEAD < 2u * 8u * kCUsPerXCD * 64u);
    bool first_requested = false;
    if(EXPLICIT && early)
    {
        const int own = GROUPS > 1 ? max(n_steps - grp + GROUPS - 1, 0) / GROUPS : n_steps;
        if(own > 0)
        {
            fetch_k(cur, lds_k0);
            fetch_v(cur, lds_v0);
            if(own > 1)
            {
                advance(nxt);
                fetch_k(nxt, lds_k1);
                nxt = cur;
            }
            first_requested = true;
        }
    }
    // Explicit masks: number of leading key steps in which the mask changes
    // nothing for any query of the workgroup (they run in the pipelined loop).
    int n_open = 0, n_skip = 0;
    if(EXPLICIT)
    {
        // The workgroup's rows of the mask are scanned once, beside the first
        // step's loads.  Per key step the scan records whether every value is
        // "open" (+0 / true) and whether every value is "hidden" (-inf /
        // false).  Hidden steps at either end are dropped - a tile pair above
        // the diagonal of a causal mask given as values costs this scan instead
        // of a pass over K and V - and open steps in front need no mask handling.
        constexpr int ES = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 2 : 1;
        constexpr uint32_t OPEN = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 0u : 0x01010101u;
        constexpr uint32_t HIDDEN = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? T::kNegInfPair : 0u;
        // bit s: some value of step s (steps >= 63 share bit 63) is not open / not hidden
        unsigned long long not_open = 0ull, not_hidden = 0ull;
        bool scanned = false;
        if(n_steps > 0 && p.mask_bits != nullptr && p.n_scan_wgs == 0)
        {
            // the scan was done once for all batch entries before the launch
            const unsigned long long *w = p.mask_bits + (int64_t)qb * (kMaskBitWords * SCAN_SPLITS);
#pragma unroll
            for(int sp = 0; sp < SCAN_SPLITS; ++sp)
            {
                uint64_t e[MaskWords::N], open, hidden;
#pragma unroll
                for(int i = 0; i < MaskWords::N; ++i)
                {
                    e[i] = w[kMaskBitWords * sp + i];
                }
                (void)MaskWords::take(e, 0u, open, hidden);
                not_open |= open;
                not_hidden |= hidden;
            }
            scanned = true;
        }
        else if(n_steps > 0 && p.mask_bits != nullptr)
        {
            // ... or is being done by the first workgroups of this launch: the
            // first wavefront waits for the entries of the block's key ranges, eight
            // lanes an entry, a word each (four entries: twice; bounded; the Q fragments are on
            // their way meanwhile), then everybody ORs.  (16 tasks of 4096 tokens, 32 heads, causal:
            // 300.4 us; 297.5 with four words an entry that were taken one by one, which
            // could be words from before; 4 % more with one lane an entry.)
            static_assert(8 % SCAN_SPLITS == 0 && kMaskBitWords <= 8, "one wavefront reads them all");
            __shared__ uint32_t got_bits[4];
            __shared__ int got_all;
            if(tid < 4)
            {
                got_bits[tid] = 0u;
            }
            __syncthreads();
            if(tid < 64)
            {
                const int i = lane & 7;
                const bool has_word = i < kMaskBitWords;
                unsigned long long *e = p.mask_bits
                    + ((int64_t)qb * SCAN_SPLITS + (lane >> 3) % SCAN_SPLITS) * kMaskBitWords
                    + (has_word ? i : 0);
                const unsigned long long t0 = wall_clock64();
                unsigned long long word;
                bool ok = true;
                for(;;)
                {
                    word = __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint64_t sum = sum_of_eight(
                            has_word ? MaskWords::share(i, word, p.mask_tag) : 0u);
                    const bool fits = !has_word
                        || (MaskWords::tagged(i, word, p.mask_tag) && sum == 0u);
                    if(__builtin_amdgcn_ballot_w64(!fits) == 0ull)
                    {
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                    if(wall_clock64() - t0 > p.mask_spin_limit)
                    {
                        ok = false;
                        break;
                    }
                }
                if(i < 4)
                {
                    atomicOr(&got_bits[i], (uint32_t)word);
                }
                if(lane == 0)
                {
                    got_all = ok;
                }
            }
            __syncthreads();
            if(got_all)
            {
                not_open = (unsigned long long)got_bits[0]
                    | ((unsigned long long)got_bits[1] << 32);
                not_hidden = (unsigned long long)got_bits[2]
                    | ((unsigned long long)got_bits[3] << 32);
                scanned = true;
            }
        }
        // (the same rows and the same bounds as in a scan done for everybody: a call's bits
        // do not depend on which of the two it has)
        if(!scanned && n_steps > 0 && k_seq * ES >= 16
                && p.mask_ld * ES * kQRows < (int64_t)(1 << 30))
        {
            __shared__ unsigned long long scan_words[2 * WAVES];
            mask_scan_steps<ES, WAVES, kKeys>(static_cast<const char *>(p.mask)
                    + (int64_t)q_row0 * p.mask_ld * ES, (uint32_t)(p.mask_ld * ES),
                    min(ROWS, q_len - q_row0), k_seq * ES, 0, (k_seq + kKeys - 1) / kKeys,
                    OPEN, HIDDEN, scan_words, not_open, not_hidden);
            scanned = true;
        }
        if(scanned)
        {
            if(not_hidden == 0ull)
            {
                if(!p.overwrite)
                {
                    // (the first step's loads may be on their way into LDS)
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    return;
                }
                n_steps = 0;    // the epilogue writes empty rows
            }
            else if((not_hidden >> 63) == 0ull)
            {
                n_steps = min(n_steps, 64 - __builtin_clzll(not_hidden));
            }
            // hidden steps at the start are passed over
            if(n_steps > 0)
            {
                n_skip = min(__builtin_ctzll(not_hidden), n_steps - 1);
            }
            not_open >>= n_skip;
            n_open = not_open == 0ull ? 63 - n_skip : min(__builtin_ctzll(not_open), 63 - n_skip);
            if(n_skip > 0)
            {
                // the step requested above is not wanted: its loads must have
                // landed before the same buffers are asked for again
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                first_requested = false;
                n_steps -= n_skip;
                cur.kb += n_skip;
                cur.rows_left -= n_skip * kKeys;
                cur.Kp += (int64_t)n_skip * kKeys * RB;
                cur.Vp += (int64_t)n_skip * kKeys * RB;
                nxt = cur;
            }
        }
    }
    // Leading steps that are complete (64 keys) and visible to every query of
    // the workgroup need no mask at all; they run in the pipelined loop below.
    int n_fast = 0;
    int n_spread = 0;       // leading steps that exist and are complete
    {
        const int n_full = (p.n_kv_tiles == 1 || k_tile % kKeys == 0)
            ? k_seq / kKeys : k_tile / kKeys;
        n_fast = min(n_steps, n_full - n_skip);
        n_spread = n_fast;
        if(MODE == NNTILE_HIP_MASK_CAUSAL)
        {
            n_fast = min(n_fast, max(rel0 + 1, 0) / kKeys);
        }
        if(EXPLICIT)
        {
            n_fast = min(n_fast, n_open);
        }
        if(GROUPS > 1)
        {
            // counted in the group's own steps (its step j is step
            // GROUPS * j + grp), and the same for both groups: the barriers of
            // the pipelined loop are the workgroup's
            n_fast /= GROUPS;
            n_spread /= GROUPS;
        }
        n_fast = n_fast >= 2 ? n_fast : 0;
    }
    // Rounds of the workgroup; from here on n_steps counts the group's own
    // steps.  A group that has one step fewer than the other goes through the
    // last round idle: every wavefront meets every barrier.
    const int n_rounds = (n_steps + GROUPS - 1) / GROUPS;
    if(GROUPS > 1)
    {
        n_steps = max(n_steps - grp + GROUPS - 1, 0) / GROUPS;
    }
    if(n_steps > 0)
    {
        if(!first_requested)
        {
            fetch_k(nxt, lds_k0);
            fetch_v(nxt, lds_v0);
        }
        advance(nxt);
        if(n_fast > 0 && !first_requested)
        {
            fetch_k(nxt, lds_k1);       // the pipelined loop keeps K two steps ahead
        }
        if(EXPLICIT && n_fast == 0)
        {
            mask_fetch(cur.kb, cur.rows_left);
        }
    }
    // ---- keys and values into this XCD's L2 ----------------------------------------
    // Workgroups of the same keys on one XCD walk them side by side, and what none of
    // them has read yet comes from HBM at every step, later than the loop asks for it
    // ahead.  So each touches a share of the lines first, four a thread at most, behind
    // its own first step's loads and where it has a step to take.  A wavefront's 64 lines
    // lie in one step of one of the two, so that where they are is scalar work and
    // nothing stands between the loads.  (Through a volatile pointer each load was waited
    // for before the next; so / now, causal, us: head 128, 25 x 1024 20.9 / 18.8, 32 x 1024 20.6 /
    // 19.2, 8 x 4096 48.8 / 46.8, 8 x 1000 14.8 / 14.2; head 64, 40 x 1000 15.2 / 14.3; masks as
    // values, head 64, 9 x 2048 25.1 / 24.0, open 30.2 / 29.2.)
    if constexpr(KH > 1)
    {
        if(p.touch_steps > 0 && n_steps > 0)
        {
            constexpr int NT = 4;
            constexpr int LINES = kKeys * RB / 128;     // of a step's K, and of its V
            static_assert(LINES % 64 == 0, "a wavefront's lines lie in one step's K or V");
            const int share = n_places * p.touch_group;
            const int idx = p.touch_group > 1
                ? my_place * p.touch_group + (b / p.n_batch) % p.touch_group : my_place;
            const int n_lines = p.touch_steps * 2 * LINES;
            uint32_t touched[NT];
#pragma unroll
            for(int i = 0; i < NT; ++i)
            {
                const int line = __builtin_amdgcn_readfirstlane((i * share + idx) * THREADS + wave * 64);
                touched[i] = 0u;
                if(line < n_lines)
                {
                    const int st = line / (2 * LINES), in = line % (2 * LINES);
                    const int kt = p.n_kv_tiles > 1 ? st / p.k_blocks_per_tile : 0;
                    const int64_t rows = min(p.k_tile, p.k_seq - kt * p.k_tile);
                    const int64_t at = min((int64_t)(st - kt * p.k_blocks_per_tile) * (kKeys * RB)
                            + (in % LINES + lane) * 128, rows * RB - 16);
                    const char *entry = static_cast<const char *>(in < LINES ? p.K[k_tile0 + kt]
                            : p.V[k_tile0 + kt]) + (int64_t)kvb * (p.kv_rows > 0 ? p.kv_rows : rows) * RB;
                    touched[i] = *(const __attribute__((address_space(1))) uint32_t *)(uintptr_t)(entry + at);
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for(int i = 0; i < NT; ++i)
            {
                asm volatile("" :: "v"(touched[i]));
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    PF_STAMP(1);
#ifdef NNTILE_PF_TRACE
    const unsigned long long pf_cycles0 = clock64();
#endif
    PF_NOTE(5, ((unsigned long long)__builtin_amdgcn_s_getreg(63508) << 32)
            | (unsigned)__builtin_amdgcn_s_getreg(63492));
    PF_NOTE(6, ((unsigned long long)(unsigned)n_steps << 32) | (unsigned)(b * 1024 + qblk));

    // One key step on LDS buffer BUF (a compile-time constant, so that every
    // LDS address is a fixed register plus an immediate).
    auto step = [&](int g, auto buf_tag) __attribute__((always_inline))
    {
        constexpr int BUF = decltype(buf_tag)::value;
        const char *Ks = BUF ? lds_k1 : lds_k0;
        const char *Vs = BUF ? lds_v1 : lds_v0;
        const int k_row0 = cur.kb * kKeys;                   // within the tile
        const int kg0 = cur.kt * k_tile + k_row0;            // key row overall
        const int keys_here = min(kKeys, cur.rows_left);
        // explicit mask: what this wavefront's block of the mask looks like
        // (the values were loaded during the previous step)
        int mask_class = MASK_MIXED;
        if(EXPLICIT)
        {
            if(keys_here < kKeys)
            {
                mask_fix_ragged(keys_here);
            }
            mask_class = mask_classify();
            if(mask_class == MASK_MIXED)
            {
                mask_transpose();
            }
        }
        // nothing of this step is visible to this wavefront, or the step is
        // the other group's last one and this group has none in this round
        const bool idle = (GROUPS > 1 && g >= n_steps)
            || (EXPLICIT ? (mask_class == MASK_HIDDEN)
            : ((MODE == NNTILE_HIP_MASK_CAUSAL) && (kg0 + kh * 32 > wave_rel_lo + 31)));

        // ---- loads of the next step into the other buffer ----------------------
        // (every wavefront passed the barrier that ended step g-1, so nobody
        // still reads that buffer)
        NNTILE_PHASE(0)
        if(g + 1 < n_steps)
        {
            fetch_k(nxt, BUF ? lds_k0 : lds_k1);
            fetch_v(nxt, BUF ? lds_v0 : lds_v1);
            advance(nxt);
        }

        uint32_t pk[NB][8];
        if(!idle)
        {
            // ---- S^T = K Q^T -------------------------------------------------
            f32x16 s[NB];
#pragma unroll
            for(int mb = 0; mb < NB; ++mb)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    s[mb][r] = 0.0f;
                }
#pragma unroll
                for(int ks = 0; ks < KSTEPS; ++ks)
                {
                    const vec8 a = *reinterpret_cast<const vec8 *>(
                            Ks + k_raddr[mb][ks]);
                    s[mb] = T::mfma(a, qf[ks], s[mb]);
                }
            }
            NNTILE_PHASE(1)

            // ---- mask ---------------------------------------------------------
            // register r of block mb holds key  (mb + kh)*32 + 8*(r/4) + 4*half + r%4
            if(EXPLICIT)
            {
                if(mask_class == MASK_MIXED)
                {
#pragma unroll
                    for(int i = 0; i < 4 * NB; ++i)
                    {
                        // group i: block i/4, registers 4*(i%4) .. +3
                        const int mb = i >> 2, r0 = 4 * (i & 3);
                        if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                        {
#pragma unroll
                            for(int e = 0; e < 4; ++e)
                            {
                                const uint32_t w = mraw[2 * i + (e >> 1)];
                                const float add = T::to_float((uint16_t)(
                                            (e & 1) ? (w >> 16) : (w & 0xffffu)));
                                s[mb][r0 + e] = fmaf(add, inv_scale, s[mb][r0 + e]);
                            }
                        }
                        else
                        {
#pragma unroll
                            for(int e = 0; e < 4; ++e)
                            {
                                if(((mraw[i] >> (8 * e)) & 0xffu) == 0u)
                                {
                                    s[mb][r0 + e] = neg_inf();
                                }
                            }
                        }
                    }
                }
            }
            else
            {
                const bool ragged = keys_here < kKeys;
                const bool diagonal = (MODE == NNTILE_HIP_MASK_CAUSAL)
                    && (kg0 + (kh + NB) * 32 - 1 > wave_rel_lo);
                if(ragged || diagonal)
                {
                    // last visible key of this step for this lane's query
                    int lim = keys_here - 1;
                    if(MODE == NNTILE_HIP_MASK_CAUSAL)
                    {
                        lim = min(lim, my_rel - kg0);
                    }
                    lim -= kh * 32;
#pragma unroll
                    for(int mb = 0; mb < NB; ++mb)
                    {
#pragma unroll
                        for(int r = 0; r < 16; ++r)
                        {
                            const int key = mb * 32 + 8 * (r >> 2) + 4 * half
                                + (r & 3);
                            if(key > lim)
                            {
                                s[mb][r] = neg_inf();
                            }
                        }
                    }
                }
            }

            // ---- online softmax -------------------------------------------------
            float mx = neg_inf();
#pragma unroll
            for(int mb = 0; mb < NB; ++mb)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    mx = fmaxf(mx, s[mb][r]);
                }
            }
            mx = max_across_halves(mx);
            const float m_new = fmaxf(m_run, mx);
            const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
            const float mc = m_use * c;
            // The running maximum rarely moves after the first steps; the
            // rescale of the 16*DBLOCKS output registers is skipped unless
            // some query of the wavefront needs it.
            if(__builtin_amdgcn_ballot_w64(m_new != m_run) != 0)
            {
                const float alpha = fast_exp2((m_run - m_use) * c);
                l_run *= alpha;
#pragma unroll
                for(int db = 0; db < DBLOCKS; ++db)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        o[db][r] *= alpha;
                    }
                }
                m_run = m_new;
            }

            // row sums by plain additions (the dot-product instruction that
            // would sum a packed pair waits for the matrix unit)
            float rs0 = 0.0f, rs1 = 0.0f;
#pragma unroll
            for(int mb = 0; mb < NB; ++mb)
            {
#pragma unroll
                for(int r = 0; r < 16; r += 2)
                {
                    const float p0 = fast_exp2(fmaf(s[mb][r], c, -mc));
                    const float p1 = fast_exp2(fmaf(s[mb][r + 1], c, -mc));
                    pk[mb][r >> 1] = T::pack2(p0, p1);
                    rs0 += p0;
                    rs1 += p1;
                }
            }
            l_run += rs0 + rs1;
        }
        // mask values of the next step (this step's have been consumed)
        if(EXPLICIT && g + 1 < n_steps)
        {
            mask_fetch(cur.kb + GROUPS, cur.rows_left - GROUPS * kKeys);
        }
        NNTILE_PHASE(2)

        // ---- O^T += V^T P^T ------------------------------------------------------
        if(!idle)
        {
#pragma unroll
            for(int t = 0; t < 2 * NB; ++t)
            {
                const int mb = t >> 1, tt = t & 1;
                const u32x4 praw = {pk[mb][4 * tt], pk[mb][4 * tt + 1],
                    pk[mb][4 * tt + 2], pk[mb][4 * tt + 3]};
                const vec8 pb = __builtin_bit_cast(vec8, praw);
#pragma unroll
                for(int db = 0; db < DBLOCKS; ++db)
                {
                    const char *src = Vs + v_raddr[db] + (16 * t) * RB;
                    const u32x2 lo = lds_read_tr16(src);
                    const u32x2 hi = lds_read_tr16(src + 8 * RB);
                    const u32x4 araw = {lo[0], lo[1], hi[0], hi[1]};
                    const vec8 a = __builtin_bit_cast(vec8, araw);
                    o[db] = T::mfma(a, pb, o[db]);
                }
            }
        }
        advance(cur);
        NNTILE_PHASE(3)
        // this wavefront's loads of the next step have landed in LDS
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        NNTILE_PHASE(4)
    };

    // ---- pipelined loop over the unmasked steps ---------------------------------
    // A step is two sub-blocks of 32 keys.  While the softmax of sub-block j
    // runs on the vector ALU, the matrix unit computes the scores of sub-block
    // j+1 and adds sub-block j-1 to the output: the three are independent, and
    // a wavefront's MFMAs execute in the background of its own VALU work.  One
    // MFMA and a slice of the softmax form a slot; scheduling barriers keep the
    // compiler from regrouping the slots.  K is fetched two steps ahead and V
    // one step ahead, with one workgroup barrier in the middle of each step.
    int g_first = 0;        // first step of the general loop
    if(n_fast > 0)
    {
        constexpr int NSLOT = 2 * KSTEPS;       // KSTEPS score MFMAs + 2*DBLOCKS output MFMAs
        constexpr int NITEM = 24;               // softmax work items of a sub-block
        constexpr float kLazyLimit = 16384.0f;  // largest row sum of a sub-block taken without a new maximum
        constexpr int AHEAD = NNTILE_PF_AHEAD;  // LDS operands are read this many slots early
        f32x16 zero16;
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            zero16[r] = 0.0f;
        }
        f32x16 sa = zero16, sb = zero16;        // scores of the current / next sub-block
        uint32_t pp[8];                         // probabilities (packed pairs) of a sub-block
#pragma unroll
        for(int i = 0; i < 8; ++i)
        {
            pp[i] = 0u;
        }
        float alpha_pending = 1.0f;             // rescale of O that the last softmax asked for
        bool rescale_pending = false;           // ... if it asked for one (the same for the whole wavefront)
        StepCursor c1 = nxt;                    // step g+1: its V is fetched during step g
        StepCursor c2 = nxt;                    // step g+2: its K is fetched during step g
        advance(c2);

        // MFMA of slot sl.  Order: first the score MFMAs (one accumulator
        // chain, which costs nothing extra), then the output MFMAs: the scores
        // are complete half a body before the next body's softmax needs them.
        //   kind 0: output MFMA number idx (16-key half idx / DBLOCKS, block idx % DBLOCKS)
        //   kind 1: score MFMA number idx (head values 16*idx .. +15)
        auto slot_kind = [](int sl) -> int
        {
            return sl < KSTEPS ? 1 : 0;
        };
        auto slot_idx = [](int sl) -> int
        {
            return sl < KSTEPS ? sl : sl - KSTEPS;
        };

        // One sub-block body.  s_cur: scores to turn into probabilities;
        // s_nxt: scores to compute from the 32 keys of block kh of buffer Kb;
        // the probabilities in pp multiply the keys 32*vh.. of buffer Vb.
        // With DO_FETCH the loads of K(c2) into kdst and V(c1) into vdst (both
        // full steps) are issued one every second slot: issued together after
        // the barrier they queue up behind each other - the loads of a step
        // take the CU's memory path about 500 cycles - and the wavefront
        // stands still until its last one is accepted.
        auto body = [&](auto do_s_tag, auto do_pv_tag, auto do_sm_tag, auto do_fetch_tag,
                const char *Kb, int kh, const char *Vb, int vh, const f32x16 &s_cur,
                f32x16 &s_nxt, char *kdst, char *vdst)
            __attribute__((always_inline))
        {
            constexpr bool DO_S = decltype(do_s_tag)::value;
            constexpr bool DO_PV = decltype(do_pv_tag)::value;
            constexpr bool DO_SM = decltype(do_sm_tag)::value;
            constexpr int DO_FETCH = decltype(do_fetch_tag)::value;    // 0, or one load every DO_FETCH slots
            static_assert(2 * LOADS_PER_WAVE * DO_FETCH <= NSLOT, "the loads fit the slots");
            auto fetch_piece = [&](int i) __attribute__((always_inline))
            {
                if(i < LOADS_PER_WAVE)
                {
                    load_to_lds16<0, false>(c2.Kp, k_goff[i], kdst + i * 1024);
                }
                else if(i < 2 * LOADS_PER_WAVE)
                {
                    switch(i - LOADS_PER_WAVE)
                    {
                        case 0: load_to_lds16<0, false>(c1.Vp, v_goff0, vdst); break;
                        case 1: load_to_lds16<1024, false>(c1.Vp, v_goff0, vdst); break;
                        case 2: load_to_lds16<2048, false>(c1.Vp, v_goff0, vdst); break;
                        default: load_to_lds16<3072, false>(c1.Vp, v_goff0, vdst); break;
                    }
                }
            };
            // the rescale that the previous softmax decided on (rare after the
            // first steps): O holds every sub-block up to j-2 at this point
            if(rescale_pending)
            {
#pragma unroll
                for(int db = 0; db < DBLOCKS; ++db)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        o[db][r] *= alpha_pending;
                    }
                }
            }
            vec8 opnd[NSLOT];       // LDS operand of each slot's MFMA
            // the probabilities of sub-block j-1, as they are on entry: pp is
            // rewritten with those of sub-block j while the output MFMAs run
            uint32_t pin[8];
#pragma unroll
            for(int i = 0; i < 8; ++i)
            {
                pin[i] = pp[i];
            }
            auto read_operand = [&](int sl) __attribute__((always_inline))
            {
                if(sl >= NSLOT)
                {
                    return;
                }
                const int i = slot_idx(sl);
                if(slot_kind(sl) == 1)
                {
                    if(DO_S)
                    {
                        opnd[sl] = *reinterpret_cast<const vec8 *>(Kb + k_raddr[0][i]
                                + kh * 32 * RB);
                    }
                }
                else if(DO_PV)
                {
                    const int t = 2 * vh + i / DBLOCKS, db = i % DBLOCKS;
                    const char *src = Vb + v_raddr[db] + (16 * t) * RB;
                    const u32x2 lo = lds_read_tr16(src);
                    const u32x2 hi = lds_read_tr16(src + 8 * RB);
                    const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                    opnd[sl] = __builtin_bit_cast(vec8, raw);
                }
            };
            // Lazy maximum: the probabilities are taken relative to the running
            // maximum as it stands, without looking at this sub-block's scores
            // first (softmax does not depend on the reference point, only
            // overflow does).  The row sums, which are needed anyway, tell
            // afterwards whether that was safe; if not (first sub-block, or
            // scores far above everything seen so far) the sub-block is redone
            // with a new maximum at the end of the body.
            const float mc = m_run * c;
            float rs = 0.0f;
            float pe[2] = {0.0f, 0.0f};
            auto item = [&](int it) __attribute__((always_inline))
            {
                const int k = it / 3, r = it % 3;
                if(r < 2)
                {
                    pe[r] = fast_exp2(fmaf(s_cur[2 * k + r], c, -mc));
                }
                else
                {
                    // (plain additions: the dot-product instruction that sums a
                    // packed pair waits for the matrix unit, 15 cycles each)
                    rs += pe[0];
                    rs += pe[1];
                    pp[k] = T::pack2(pe[0], pe[1]);
                    // (keeps the conversion in this slot)
                    asm volatile("" : "+v"(pp[k]));
                }
            };
#pragma unroll
            for(int sl = 0; sl < AHEAD; ++sl)
            {
                read_operand(sl);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for(int sl = 0; sl < NSLOT; ++sl)
            {
                read_operand(sl + AHEAD);
                const int i = slot_idx(sl);
                if(slot_kind(sl) == 1)
                {
                    if(DO_S)
                    {
                        s_nxt = T::mfma(opnd[sl], qf[i], i == 0 ? zero16 : s_nxt);
                    }
                }
                else if(DO_PV)
                {
                    const int t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x4 praw = {pin[4 * t], pin[4 * t + 1], pin[4 * t + 2],
                        pin[4 * t + 3]};
                    o[db] = T::mfma(opnd[sl], __builtin_bit_cast(vec8, praw), o[db]);
                }
                // the softmax items are spread over the slots 1 .. NSLOT-1
                if(DO_SM && sl >= 1)
                {
#pragma unroll
                    for(int it = (sl - 1) * NITEM / (NSLOT - 1);
                            it < sl * NITEM / (NSLOT - 1); ++it)
                    {
                        item(it);
                    }
                }
                if(DO_FETCH > 0 && sl % max(DO_FETCH, 1) == DO_FETCH - 1)
                {
                    fetch_piece(sl / max(DO_FETCH, 1));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            rescale_pending = false;
            if(DO_SM)
            {
                if(__builtin_amdgcn_ballot_w64(!(rs <= kLazyLimit)) != 0)
                {
                    float mx = s_cur[0];
#pragma unroll
                    for(int r = 1; r < 16; ++r)
                    {
                        mx = fmaxf(mx, s_cur[r]);
                    }
                    // every key of these steps is visible: the new maximum is finite
                    const float m_new = max_with_other_half(m_run, mx);
                    const float alpha = fast_exp2((m_run - m_new) * c);
                    const float mc_new = m_new * c;
                    rs = 0.0f;
#pragma unroll
                    for(int k = 0; k < 8; ++k)
                    {
                        const float p0 = fast_exp2(fmaf(s_cur[2 * k], c, -mc_new));
                        const float p1 = fast_exp2(fmaf(s_cur[2 * k + 1], c, -mc_new));
                        pp[k] = T::pack2(p0, p1);
                        rs += p0;
                        rs += p1;
                    }
                    l_run *= alpha;
                    m_run = m_new;
                    alpha_pending = alpha;
                    rescale_pending = true;
                }
                l_run += rs;
            }
            // Everything above belongs to this body: without this the compiler
            // sinks the tail of the softmax, whose results are first used by
            // the next body, behind that body's rescale branch and out of the
            // shadow of the MFMAs.
            asm volatile("" : "+v"(pp[0]), "+v"(pp[1]), "+v"(pp[2]), "+v"(pp[3]),
                    "+v"(pp[4]), "+v"(pp[5]), "+v"(pp[6]), "+v"(pp[7]),
                    "+v"(l_run), "+v"(m_run));
            if(DO_S)
            {
                asm volatile("" : "+v"(s_nxt));
            }
        };
        typedef std::integral_constant<bool, true> Yes;
        typedef std::integral_constant<bool, false> No;
        typedef std::integral_constant<int, 0> NoFetch;
        typedef std::integral_constant<int, (KH > 1 ? 1 : 2)> Spread;

        // scores of sub-block (0, 0)
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            const vec8 a = *reinterpret_cast<const vec8 *>(lds_k0 + k_raddr[0][ks]);
            sa = T::mfma(a, qf[ks], ks == 0 ? zero16 : sa);
        }

        // The middle of step g on the buffers of parity BUF: K(g+1) and V(g)
        // have landed for everyone (they were requested a step ago) and nobody
        // reads K(g) or V(g-1) any more, so their buffers take K(g+2), V(g+1).
        auto mid_step = [&](int g, auto buf_tag) __attribute__((always_inline))
        {
            constexpr int BUF = decltype(buf_tag)::value;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if(g + 2 < n_steps)
            {
                fetch_k(c2, BUF ? lds_k1 : lds_k0);
            }
            if(g + 1 < n_steps)
            {
                fetch_v(c1, BUF ? lds_v0 : lds_v1);
            }
            c1 = c2;
            advance(c2);
        };
        char *const no_dst = nullptr;
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        // One step on the buffers of parity BUF: sub-block (g, 0) with the
        // scores of (g, 1) and the output of (g-1, 1), then sub-block (g, 1)
        // with the scores of (g+1, 0) and the output of (g, 0).  (After the
        // last pipelined step the scores computed ahead are not used.)
        // spread_tag: steps g+1 and g+2 exist and are complete, and their
        // loads go into the slots of the second sub-block.
        auto fast_step = [&](int g, auto buf_tag, auto spread_tag) __attribute__((always_inline))
        {
            constexpr int BUF = decltype(buf_tag)::value;
            body(Yes{}, Yes{}, Yes{}, NoFetch{}, BUF ? lds_k1 : lds_k0, 1, BUF ? lds_v0 : lds_v1, 1,
                    sa, sb, no_dst, no_dst);
            if(decltype(spread_tag)::value)
            {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                char *kdst = (BUF ? lds_k1 : lds_k0) + lds_grp_off + wave_u * LOADS_PER_WAVE * 1024;
                char *vdst = (BUF ? lds_v0 : lds_v1) + lds_grp_off + wave_u * LOADS_PER_WAVE * 1024;
                body(Yes{}, Yes{}, Yes{}, Spread{}, BUF ? lds_k0 : lds_k1, 0,
                        BUF ? lds_v1 : lds_v0, 0, sb, sa, kdst, vdst);
                c1 = c2;
                advance(c2);
            }
            else
            {
                mid_step(g, buf_tag);
                body(Yes{}, Yes{}, Yes{}, NoFetch{}, BUF ? lds_k0 : lds_k1, 0,
                        BUF ? lds_v1 : lds_v0, 0, sb, sa, no_dst, no_dst);
            }
            advance(cur);
        };
        if constexpr(KH > 1)
        {
            // A step is one sub-block of every wavefront: body g takes the softmax of
            // step g, the scores of step g+1 and the output of step g-1.  K(g+2) takes
            // the buffer of K(g), whose scores were taken a body ago, and V(g) the one
            // of V(g-2); both are waited for at the end of the body.
            auto end_body = [&]() __attribute__((always_inline))
            {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                advance(cur);
            };
            auto one_step = [&](int g, auto buf_tag, auto spread_tag) __attribute__((always_inline))
            {
                constexpr int BUF = decltype(buf_tag)::value;
                char *kbuf = BUF ? lds_k1 : lds_k0, *vbuf = BUF ? lds_v1 : lds_v0;
                const char *k_next = BUF ? lds_k0 : lds_k1, *v_prev = BUF ? lds_v0 : lds_v1;
                f32x16 &s_cur = BUF ? sb : sa, &s_nxt = BUF ? sa : sb;
                if(decltype(spread_tag)::value)
                {
                    const int at = wave_u * LOADS_PER_WAVE * 1024;
                    c1 = cur;
                    body(Yes{}, Yes{}, Yes{}, Spread{}, k_next, 0, v_prev, 0, s_cur, s_nxt,
                            kbuf + at, vbuf + at);
                    advance(c2);
                }
                else
                {
                    fetch_v(cur, vbuf);
                    if(g + 2 <= n_fast && g + 2 < n_steps)
                    {
                        fetch_k(c2, kbuf);
                        advance(c2);
                    }
                    body(Yes{}, Yes{}, Yes{}, NoFetch{}, k_next, 0, v_prev, 0, s_cur, s_nxt,
                            no_dst, no_dst);
                }
                end_body();
            };
            // (every wavefront has taken the scores of step 0)
            __syncthreads();
            if(2 <= n_fast && 2 < n_steps)
            {
                fetch_k(c2, lds_k0);
                advance(c2);
            }
            body(Yes{}, No{}, Yes{}, NoFetch{}, lds_k1, 0, lds_v0, 0, sa, sb, no_dst, no_dst);
            end_body();
            int g = 1;
            for(; g + 3 <= n_fast && g + 3 < n_spread; g += 2)
            {
                one_step(g, std::integral_constant<int, 1>{}, Yes{});
                one_step(g + 1, std::integral_constant<int, 0>{}, Yes{});
            }
            for(; g < n_fast; g += 2)
            {
                one_step(g, std::integral_constant<int, 1>{}, No{});
                if(g + 1 < n_fast)
                {
                    one_step(g + 1, std::integral_constant<int, 0>{}, No{});
                }
            }
            // cur is step n_fast now; its K is there where the general loop takes it
            // up, its V takes the buffer of V(n_fast-2)
            if(n_fast < n_steps)
            {
                fetch_v(cur, (n_fast & 1) ? lds_v1 : lds_v0);
            }
            c1 = cur;
            advance(c1);
        }
        else
        {
            // step 0: there is no output yet in its first half
            body(Yes{}, No{}, Yes{}, NoFetch{}, lds_k0, 1, lds_v1, 1, sa, sb, no_dst, no_dst);
            mid_step(0, std::integral_constant<int, 0>{});
            body(Yes{}, Yes{}, Yes{}, NoFetch{}, lds_k1, 0, lds_v0, 0, sb, sa, no_dst, no_dst);
            advance(cur);
            int g = 1;
            for(; g + 1 < n_fast && g + 3 < n_spread; g += 2)
            {
                fast_step(g, std::integral_constant<int, 1>{}, Yes{});
                fast_step(g + 1, std::integral_constant<int, 0>{}, Yes{});
            }
            // the last steps, whose successors may be incomplete or absent
            for(; g < n_fast; g += 2)
            {
                fast_step(g, std::integral_constant<int, 1>{}, No{});
                if(g + 1 < n_fast)
                {
                    fast_step(g + 1, std::integral_constant<int, 0>{}, No{});
                }
            }
        }
        if(EXPLICIT && n_fast < n_steps)
        {
            mask_fetch(cur.kb, cur.rows_left);     // the general step finds its mask values loaded
        }
        // drain: the output of the last sub-block
        if((n_fast - 1) & 1)
        {
            body(No{}, Yes{}, No{}, NoFetch{}, lds_k0, 0, lds_v1, NB - 1, sb, sa, no_dst, no_dst);
        }
        else
        {
            body(No{}, Yes{}, No{}, NoFetch{}, lds_k0, 0, lds_v0, NB - 1, sb, sa, no_dst, no_dst);
        }
        g_first = n_fast;
        nxt = c1;
        // the general loop expects step g_first complete in its buffers
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    PF_STAMP(2);
    {
        int g = g_first;
        if(g < n_rounds && (g & 1))
        {
            step(g, std::integral_constant<int, 1>{});
            g += 1;
        }
        for(; g < n_rounds; g += 2)
        {
            step(g, std::integral_constant<int, 0>{});
            if(g + 1 < n_rounds)
            {
                step(g + 1, std::integral_constant<int, 1>{});
            }
        }
    }
    NNTILE_PHASE_DUMP()
    PF_STAMP(3);
    PF_NOTE(7, clock64() - pf_cycles0);     // shader-clock cycles between stamps 1 and 3

    // ---- the second group hands its triple to the first -------------------------
    // Through the K/V arrays, which nobody reads any more: wavefront w of the
    // second group writes (O, maximum, sum) lane by lane into array w, its
    // counterpart in the first group - same queries, same lanes - combines
    // them with its own as two partial softmaxes are combined.
    if constexpr(GROUPS > 1)
    {
        constexpr int NO = 16 * DBLOCKS;
        static_assert(GROUPS == 1 || (NO + 2) * 256 <= K_BYTES * GROUPS - 32 * RB,
                "the triple and the epilogue's staging rows share an array");
        float *mrg = reinterpret_cast<float *>(wave == 0 ? lds_k0 : wave == 1 ? lds_k1
                : wave == 2 ? lds_v0 : lds_v1) + lane;
        __syncthreads();
        if(grp == 1)
        {
#pragma unroll
            for(int db = 0; db < DBLOCKS; ++db)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    mrg[(16 * db + r) * 64] = o[db][r];
                }
            }
            mrg[NO * 64] = m_run;
            mrg[(NO + 1) * 64] = l_run;
        }
        __syncthreads();
        if(grp == 1)
        {
            return;
        }
        const float m_other = mrg[NO * 64];
        const float l_other = mrg[(NO + 1) * 64];
        const float m_new = fmaxf(m_run, m_other);
        // (a group that saw no visible key has maximum -inf and weight 0)
        const float a_mine = (m_run == neg_inf()) ? 0.0f : fast_exp2((m_run - m_new) * c);
        const float a_other = (m_other == neg_inf()) ? 0.0f : fast_exp2((m_other - m_new) * c);
#pragma unroll
        for(int db = 0; db < DBLOCKS; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o[db][r] = o[db][r] * a_mine + mrg[(16 * db + r) * 64] * a_other;
            }
        }
        l_run = l_run * a_mine + l_other * a_other;
        m_run = m_new;
    }

    // ---- the two halves of a step's keys are put together ------------------------
    // Wavefronts w and w + 2 hold the same queries: each writes the half of its output
    // that the other is left with, and takes its own.
    if constexpr(KH > 1)
    {
        static_assert((16 * NDB + 2) * 256 <= K_BYTES - 32 * RBE,
                "the triple and the epilogue's staging rows share an array");
        auto array = [&](int w) __attribute__((always_inline)) -> char *
        {
            return w == 0 ? lds_k0 : w == 1 ? lds_k1 : w == 2 ? lds_v0 : lds_v1;
        };
        float *mine = reinterpret_cast<float *>(array(wave)) + lane;
        const float *theirs = reinterpret_cast<const float *>(array(wave ^ 2)) + lane;
#pragma unroll
        for(int db = 0; db < NDB; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                mine[(16 * db + r) * 64] = o[NDB + db][r];
            }
        }
        mine[16 * NDB * 64] = m_run;
        mine[(16 * NDB + 1) * 64] = l_run;
        __syncthreads();
        const float m_other = theirs[16 * NDB * 64];
        const float l_other = theirs[(16 * NDB + 1) * 64];
        const float m_new = fmaxf(m_run, m_other);
        // (a half that saw no visible key has maximum -inf and weight 0)
        const float a_mine = (m_run == neg_inf()) ? 0.0f : fast_exp2((m_run - m_new) * c);
        const float a_other = (m_other == neg_inf()) ? 0.0f : fast_exp2((m_other - m_new) * c);
#pragma unroll
        for(int db = 0; db < NDB; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o[db][r] = o[db][r] * a_mine + theirs[(16 * db + r) * 64] * a_other;
            }
        }
        l_run = l_run * a_mine + l_other * a_other;
        m_run = m_new;
    }

    // ---- epilogue: normalise, merge into the running (lse, A) ----------------
    const float l_tot = sum_across_halves(l_run);
    // no visible key for this query.  A score that is NaN makes the sum NaN: such
    // a row is NaN where (lse, A) are overwritten, and is not merged into a
    // running pair (src/kernel/accumulate_attn_output/cuda.cu:43-50).
    const bool empty = l_tot == 0.0f;
    if constexpr(PARTS)
    {
        if(q_ok)
        {
            // (a sum that is NaN goes out as it is, with some finite maximum)
            const int64_t row = ((int64_t)part * p.batch + b) * p.q_seq + my_q;
            if(half == 0)
            {
                p.part_ml[2 * row] = empty ? neg_inf() : l_tot > 0.0f ? m_run * p.scale : 0.0f;
                p.part_ml[2 * row + 1] = l_tot;
            }
            float *dst = p.part_o + row * HEAD + 4 * half;
#pragma unroll
            for(int db = 0; db < DBLOCKS; ++db)
            {
#pragma unroll
                for(int rg = 0; rg < 4; ++rg)
                {
                    f32x4 v;
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                    {
                        v[e] = empty ? 0.0f : o[db][4 * rg + e];
                    }
                    *reinterpret_cast<f32x4 *>(dst + 32 * db + 8 * rg) = v;
                }
            }
        }
        return;
    }
    // rows that are written; the others leave lse and A as they are
    const bool live = q_ok && (l_tot > 0.0f || p.overwrite);
    const float to_ln = p.scale;
    const float lse_new = empty ? neg_inf() : m_run * to_ln + __logf(l_tot);
    const float lse_old = live ? lse_stored : neg_inf();
    float w_old = 0.0f, w_new = 0.0f, lse_out = neg_inf();
    if(live && !empty)
    {
        merge_weights(lse_old, lse_new, w_old, w_new, lse_out);
    }
    if(live && half == 0 && kh == 0)
    {
        *lse_ptr = lse_out;
    }
    const float w_o = (empty || !live) ? 0.0f : w_new / l_tot;
    // register r of block db holds head value  db*32 + 8*(r/4) + 4*half + r%4

    // The wavefront's 32 rows go through LDS (its own quarter of the K
    // buffers, which nobody reads any more after the last barrier) so that they
    // leave as whole rows, 16 bytes per lane, instead of 8-byte pieces 2*HEAD
    // bytes apart - and, where the old A is merged in, come the same way: all
    // its loads are in flight at once and a lane finds its pieces where it
    // writes the sums.  (Loaded and stored in 8-byte pieces the merge of a
    // 1024 x 1024 x 32 tile pair took 3 us more.)
    // 16-byte chunk c of row r sits at chunk position c ^ (r % CPR).
    // (two wavefronts per buffer: K0, K1, then V0, V1 for wavefronts 4 to 7)
    // (two groups: wavefront w uses the end of array w, behind the triple
    // it has just read - a neighbour may still be reading its own)
    char *xch = GROUPS > 1
        ? (wave == 0 ? lds_k0 : wave == 1 ? lds_k1 : wave == 2 ? lds_v0 : lds_v1)
            + (K_BYTES * GROUPS - 32 * RB)
        : KH > 1 ? (wave == 0 ? lds_k0 : wave == 1 ? lds_k1 : wave == 2 ? lds_v0 : lds_v1)
            + (K_BYTES - 32 * RBE)
        : ((wave >> 1) == 0 ? lds_k0 : (wave >> 1) == 1 ? lds_k1
            : (wave >> 1) == 2 ? lds_v0 : lds_v1) + (wave & 1) * 32 * RB;
    const uint64_t live_rows = __builtin_amdgcn_ballot_w64(live && half == 0);
    constexpr int ROWS_PER_ST = 1024 / RBE;     // rows one load or store instruction covers
    constexpr int N_ST = 32 / ROWS_PER_ST;
    const int st_row = lane / CPRE, st_c = lane % CPRE;
    char *Abase = static_cast<char *>(p.A[q_tile0 + qt])
        + ((int64_t)b * q_len + q_row0 + rb * 32) * RB + kh * RBE;
    const bool merge = __builtin_amdgcn_ballot_w64(live && w_old != 0.0f) != 0;
    if(merge)
    {
        u32x4 old[N_ST];
#pragma unroll
        for(int i = 0; i < N_ST; ++i)
        {
            // (the rows of a tile end at q_len: rows past it re-read row 0)
            const int r = i * ROWS_PER_ST + st_row;
            const bool there = (live_rows >> r) & 1;
            old[i] = *reinterpret_cast<const u32x4 *>(
                    Abase + (there ? (int64_t)r * RB : -(int64_t)rb * 32 * RB) + st_c * 16);
        }
#pragma unroll
        for(int i = 0; i < N_ST; ++i)
        {
            const int r = i * ROWS_PER_ST + st_row;
            *reinterpret_cast<u32x4 *>(xch + r * RBE + (st_c ^ (r % CPRE)) * 16) = old[i];
        }
    }
#pragma unroll
    for(int db = 0; db < NDB; ++db)
    {
#pragma unroll
        for(int rg = 0; rg < 4; ++rg)
        {
            const int cpos = (db * 4 + rg) ^ (col % CPRE);
            u32x2 *at = reinterpret_cast<u32x2 *>(xch + col * RBE + cpos * 16 + 8 * half);
            float v[4];
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                v[e] = o[db][4 * rg + e] * w_o;
            }
            if(merge)
            {
                const u32x2 prev = *at;
                // (a row that does not need its old A may hold anything)
                const u32x2 old = w_old != 0.0f ? prev : u32x2{0, 0};
                v[0] += w_old * T::to_float((uint16_t)(old[0] & 0xffffu));
                v[1] += w_old * T::to_float((uint16_t)(old[0] >> 16));
                v[2] += w_old * T::to_float((uint16_t)(old[1] & 0xffffu));
                v[3] += w_old * T::to_float((uint16_t)(old[1] >> 16));
            }
            u32x2 out;
            out[0] = T::pack2(v[0], v[1]);
            out[1] = T::pack2(v[2], v[3]);
            *at = out;
        }
    }
#pragma unroll
    for(int i = 0; i < N_ST; ++i)
    {
        const int r = i * ROWS_PER_ST + st_row;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(
                xch + r * RBE + (st_c ^ (r % CPRE)) * 16);
        if((live_rows >> r) & 1)
        {
            *reinterpret_cast<u32x4 *>(Abase + (int64_t)r * RB + st_c * 16) = v;
        }
    }
#ifdef NNTILE_PF_TRACE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    PF_STAMP(4);
#endif
}

template<typename T, int HEAD>
static int launch_mode(hipStream_t stream, const PrefillParams &p, int mode,
        dim3 grid, bool wide, bool key_split, bool halved)
{
    if constexpr(HEAD >= 64)
    {
        if(halved)
        {
            auto launch = [&](auto kernel) -> int
            {
                hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, p);
                return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
            };
            switch(mode)
            {
                case NNTILE_HIP_MASK_ADDITIVE:
                    return launch(sdpa_prefill_16bit_kernel<T, HEAD, NNTILE_HIP_MASK_ADDITIVE, 4, 1, false, 2>);
                case NNTILE_HIP_MASK_NONE:
                    return launch(sdpa_prefill_16bit_kernel<T, HEAD, NNTILE_HIP_MASK_NONE, 4, 1, false, 2>);
                case NNTILE_HIP_MASK_CAUSAL:
                    return launch(sdpa_prefill_16bit_kernel<T, HEAD, NNTILE_HIP_MASK_CAUSAL, 4, 1, false, 2>);
                case NNTILE_HIP_MASK_BOOL:
                    return launch(sdpa_prefill_16bit_kernel<T, HEAD, NNTILE_HIP_MASK_BOOL, 4, 1, false, 2>);
                default:
                    return NNTILE_HIP_EINVAL;
            }
        }
        if(key_split)
        {
            switch(mode)
            {
                case NNTILE_HIP_MASK_ADDITIVE:
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_ADDITIVE, 8, 2>), grid, dim3(512), 0, stream, p);
                    break;
                case NNTILE_HIP_MASK_NONE:
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_NONE, 8, 2>), grid, dim3(512), 0, stream, p);
                    break;
                case NNTILE_HIP_MASK_CAUSAL:
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_CAUSAL, 8, 2>), grid, dim3(512), 0, stream, p);
                    break;
                case NNTILE_HIP_MASK_BOOL:
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_BOOL, 8, 2>), grid, dim3(512), 0, stream, p);
                    break;
                default:
                    return NNTILE_HIP_EINVAL;
            }
            return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
        }
    }
    switch(mode)
    {
        case NNTILE_HIP_MASK_ADDITIVE:
            hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                        NNTILE_HIP_MASK_ADDITIVE>), grid, dim3(kThreads), 0,
                    stream, p);
            break;
        case NNTILE_HIP_MASK_NONE:
            if constexpr(HEAD >= 64)
            {
                if(wide)
                {
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_NONE, 8>), grid, dim3(512), 0, stream, p);
                    break;
                }
            }
            hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                        NNTILE_HIP_MASK_NONE>), grid, dim3(kThreads), 0,
                    stream, p);
            break;
        case NNTILE_HIP_MASK_CAUSAL:
            if constexpr(HEAD >= 64)
            {
                if(wide)
                {
                    hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                                NNTILE_HIP_MASK_CAUSAL, 8>), grid, dim3(512), 0, stream, p);
                    break;
                }
            }
            hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                        NNTILE_HIP_MASK_CAUSAL>), grid, dim3(kThreads), 0,
                    stream, p);
            break;
        case NNTILE_HIP_MASK_BOOL:
            hipLaunchKernelGGL((sdpa_prefill_16bit_kernel<T, HEAD,
                        NNTILE_HIP_MASK_BOOL>), grid, dim3(kThreads), 0,
                    stream, p);
            break;
        default:
            return NNTILE_HIP_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

// The scan of an explicit mask that every workgroup of the attention kernel
// would do for its own rows, done once for all batch entries, as a launch
// of its own (calls under stream capture; otherwise the scan rides in the
// attention launch): workgroup (query block, key range) writes what it finds
// to entry blockIdx.x of the table (see PrefillParams::mask_bits), without a tag.
template<int ES, int ROWS>
__global__ __launch_bounds__(kThreads)
void mask_step_bits_kernel(const char *mask, uint32_t ld_bytes, int q_len, int k_seq,
        uint32_t open_word, uint32_t hidden_word, unsigned long long *table)
{
    __shared__ unsigned long long words[2 * kThreads / 64];
    unsigned long long not_open, not_hidden;
    mask_scan_range<ES, kThreads / 64, ROWS>(mask, ld_bytes, q_len, k_seq, open_word, hidden_word,
            (int)blockIdx.x / kScanSplits<ROWS>, (int)blockIdx.x % kScanSplits<ROWS>, words, not_open,
            not_hidden);
    mask_words_publish(table + kMaskBitWords * (int64_t)blockIdx.x, (int)threadIdx.x, not_open,
            not_hidden, 0ull);
}

// Masks below this size are scanned by the attention kernel's workgroups
// themselves, each its own rows, on a stream that is being captured: the shared scan
// is a launch of its own there, 2 to 3 us.  (Elsewhere it is the faster one at every
// size: 4 x 128^2 of head 64, causal, 9.1 -> 8.5 us, 30 x 256^2 of head 128 14.3 -> 13.4,
// 40 x 355^2 of head 64 15.1 -> 12.9, 40 x 430^2 of head 128 16.7 -> 15.5.)
constexpr int64_t kMaskScanBytes = 3 << 17;

// A value that no earlier call of this process has used (see MaskWords).
static uint64_t next_scan_tag()
{
    static const uint64_t start = []
    {
        std::random_device rd;
        return ((uint64_t)rd() << 32) | rd();
    }();
    static std::atomic<uint64_t> counter{0};
    return MaskWords::tag(start, counter.fetch_add(1, std::memory_order_relaxed));
}

// One-tile calls with an explicit mask and a scratch buffer of the caller's
// (the reference's scratch_logsumexp tile): scan the mask once, into the
// scratch, instead of once per batch entry - by the first workgroups of the
// attention launch itself, or, on a stream that is being captured (a replay
// would carry this call's tag again and find the words of the replay before
// it), by a launch of its own.  Leaves p.mask_bits null when the conditions of
// the kernel's own scan do not hold or the scratch is too small.  halved: the attention
// workgroups have 64 rows, and so have the scan's blocks.
template<typename T>
static int scan_mask_once(hipStream_t stream, PrefillParams &p, int mode, bool halved,
        void *scratch, size_t scratch_bytes)
{
    p.n_scan_wgs = 0;
    const bool additive = mode == NNTILE_HIP_MASK_ADDITIVE;
    if((!additive && mode != NNTILE_HIP_MASK_BOOL) || scratch == nullptr
            || p.n_q_tiles != 1 || p.n_kv_tiles != 1 || p.mask == nullptr)
    {
        return NNTILE_HIP_OK;
    }
    const int64_t es = additive ? 2 : 1;
    const int64_t row_bytes = p.k_seq * es;
    // (blocks of 64 rows take no more room: what a scratch is good for is one rule)
    const int64_t table_bytes = (p.q_seq + kQRows - 1) / kQRows * kMaskBitSplits
        * (kMaskBitWords * (int64_t)sizeof(unsigned long long));
    if(row_bytes < 16 || p.mask_ld * es * kQRows >= (int64_t)(1 << 30)
            || reinterpret_cast<uintptr_t>(scratch) % 8 != 0
            || (int64_t)scratch_bytes < table_bytes)
    {
        return NNTILE_HIP_OK;
    }
    auto *table = static_cast<unsigned long long *>(scratch);
    constexpr int kHalf = kQRows / 2;
    const int64_t n_scan = halved ? (p.q_seq + kHalf - 1) / kHalf * kScanSplits<kHalf>
        : (p.q_seq + kQRows - 1) / kQRows * kScanSplits<kQRows>;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if(hipStreamIsCapturing(stream, &capturing) != hipSuccess)
    {
        (void)hipGetLastError();
        capturing = hipStreamCaptureStatusActive;       // the careful form
    }
    if(capturing != hipStreamCaptureStatusNone
            && (p.q_seq * row_bytes < kMaskScanBytes || p.batch < 2))
    {
        return NNTILE_HIP_OK;
    }
    if(capturing == hipStreamCaptureStatusNone)
    {
        p.mask_bits = table;
        p.n_scan_wgs = (int32_t)((n_scan + 7) / 8 * 8);
        p.mask_tag = next_scan_tag();
        // A scan takes 2 us, or what 128 rows of an eighth of the keys (64 of a
        // quarter) take a workgroup: well below a byte of a row a tick of the 100 MHz clock.  Words that
        // are not there then were overwritten, by a call on another stream that
        // was lent the same memory.
        p.mask_spin_limit = 2000ull + (unsigned long long)row_bytes;
        return NNTILE_HIP_OK;
    }
    auto launch = [&](auto kernel, uint32_t open_word, uint32_t hidden_word)
    {
        hipLaunchKernelGGL(kernel, dim3((unsigned)n_scan), dim3(kThreads), 0, stream,
                static_cast<const char *>(p.mask), (uint32_t)(p.mask_ld * es), (int)p.q_seq,
                (int)p.k_seq, open_word, hidden_word, table);
    };
    if(additive)
    {
        launch(halved ? mask_step_bits_kernel<2, kHalf> : mask_step_bits_kernel<2, kQRows>, 0u,
                T::kNegInfPair);
    }
    else
    {
        launch(halved ? mask_step_bits_kernel<1, kHalf> : mask_step_bits_kernel<1, kQRows>, 0x01010101u,
                0u);
    }
    if(hipGetLastError() != hipSuccess)
    {
        return NNTILE_HIP_ELAUNCH;
    }
    p.mask_bits = table;
    return NNTILE_HIP_OK;
}

// Key steps an entry of the batch has.
static int64_t key_steps(const PrefillParams &p)
{
    const int64_t last_keys = p.k_seq - (p.n_kv_tiles - 1) * p.k_tile;
    return (p.n_kv_tiles - 1) * ((p.k_tile + kKeys - 1) / kKeys) + (last_keys + kKeys - 1) / kKeys;
}

// How the keys of a launch lie on the XCDs: `fit` leading key steps of all entries that an
// XCD works on have room in 3 of its L2's 4 MiB; `group` heads of an XCD share their keys.
// (Asked for only where the rules below need it: a call of a small tile is bound by
// the host, which its dozens of divisions would keep.)
struct KeysOnXCD
{
    int64_t fit;
    int group;
};

static KeysOnXCD keys_on_xcd(const PrefillParams &p, int head)
{
    KeysOnXCD r;
    const int64_t batch_all = (int64_t)p.batch * p.n_slabs;
    const int64_t q_blocks = (p.q_tile + kQRows / 2 - 1) / (kQRows / 2) * p.n_q_tiles;
    int64_t entries = batch_all / 8;
    r.group = 1;
    if(batch_all % 8 == 0)
    {
        if(p.n_slabs == 1 && p.batch % (8 * (int64_t)p.n_batch * p.kv_group) == 0)
        {
            r.group = p.kv_group;
        }
    }
    else
    {
        // (runs of the workgroups, as the kernel cuts them)
        const int64_t n = batch_all * q_blocks;
        for(int64_t x = 0; x < 8; ++x)
        {
            const int64_t lo = x * (n / 8) + std::min(x, n % 8);
            const int64_t hi = lo + n / 8 + (x < n % 8 ? 1 : 0);
            entries = hi > lo ? std::max(entries, (hi - 1) / q_blocks - lo / q_blocks + 1) : entries;
        }
    }
    r.fit = ((int64_t)3 << 20) * r.group / (std::max<int64_t>(entries, 1) * (kKeys * 2 * 2) * head);
    return r;
}

// From how many key steps on the first touch of the keys pays (us, touched / not, inputs
// of other calls in between; bf16, causal): head 128, 8 entries of 1024 keys 14.6 / 15.3 (without
// a mask 15.0 / 15.7), 8 x 2048 23.3 / 26.1, 4 x 4096 39.1 / 45.4, 16 x 2048 28.8 / 30.1; head 64, 24 x
// 1300 16.3 / 17.0, 8 x 4096 34.5 / 37.1, its mask as values 40.5 / 51.5.  From fewer steps on some
// lose: 12 x 300 of head 64 8.2 / 7.7, 12 x 800 12.1 / 11.5, head 128 30 x 900 20.8 / 19.6, 36 x 500
// 13.6 / 13.0, 8 x 700 12.4 / 12.6.
constexpr int64_t kTouchSteps = 16;
// ... with masks given as values and more than 256 workgroups at head 128: 24 x 1024
// without a hidden key 26.7 / 25.4, 16 x 1500 causal 25.2 / 26.6, open 33.9 / 32.7, a window 16.1 / 15.9,
// 16 x 2048 32.0 / 32.6, 45.7 / 44.5, 19.1 / 18.3
constexpr int64_t kTouchStepsMask = 24;

// Steps from which rectangular calls with an analytic mask may be halved (see below)
constexpr int64_t kHalvedSteps = 8;

// Workgroups of 64 queries whose wavefronts halve the key steps between them: twice the
// workgroups with half of the chain each, on CUs that would stand empty, or two on a CU,
// long beside short (causal); but each step comes into LDS twice as often for its MFMAs, and with
// two such workgroups a CU and no mask that is what bounds the launch.
//
// The rule, in workgroups of 64 queries:
//   up to 256         all launches, but long open ones whose keys outgrow the L2
//   257 to about 512  (at most 256 of 128 queries) not without a mask; causal by rule where it hides
//                     enough and the keys fit the L2; masks as values: head 64, and from
//                     24 steps on, where the keys fit it, both heads
//   to 768, head 64   three fit a CU: under a mask, entries in eights; other numbers of
//                     entries only the longest causal rows
// but for one line that is not there for speed: rectangular calls by rule of fewer than 8 steps
// give equal bits whatever number of entries shares their launch, which a test of this
// repository holds them to (test_gpu_backward_wide_keys.py, through the output that the
// gradients start from), although a call's last bit may otherwise depend on that.
//
// us, 128-query forms / halved, bf16, inputs of other calls in between:
//   up to 256, head 128: 8 x 128 causal 8.1 / 6.8, 4 x 300 11.7 / 9.0, 8 x 500 15.1 / 10.6, 8 x 1024 19.9 /
//   14.6, 8 x 2048 30.8 / 23.3, open 31.1 / 24.9, 4 x 4096 50.5 / 38.6, open 51.3 / 44.3; head 64: 8 x 500
//   10.6 / 8.9, 4 x 4096 37.0 / 30.4; masks as values, causal, open, window, hidden: head 128, 8 x 1024
//   23.8 22.7 16.0 4.3 / 17.3 17.5 12.2 4.4, 8 x 2048 36.0 36.8 18.9 6.1 / 27.3 29.3 14.6 6.0, 32 x 500
//   18.4 18.2 16.2 4.3 / 15.1 15.8 13.0 4.3; head 64, 12 x 1000 20.6 20.3 13.8 4.5 / 15.2 16.0 11.0
//   4.4.  Not where the keys of an open launch outgrow the L2: 1 x 16384 171.6 / 177.3.
//   257 to 512, causal: head 128, 32 x 700 17.0 / 14.6, 32 x 1024 22.2 / 19.2, 8 x 4096 54.3 / 46.8, 12 x 2048
//   31.0 / 25.0, 25 x 1024 23.3 / 18.8, 36 x 500 16.0 / 12.7, 200 x 128 10.1 / 9.5; head 64, 20 x 1500
//   19.5 / 16.5, 8 x 4096 38.3 / 32.9; up to 768 40 x 1000 18.0 / 14.3, 24 x 2000 29.2 / 23.5, 12 x 4096 50.0 /
//   41.9, 96 x 330 10.9 / 9.5, 104 x 330 11.2 / 9.8, but 100 x 330 11.4 / 11.7 and 33 x 1300 22.7 / 23.2 before
//   the touch was one batch.  4 x 8192 of head 128, whose keys outgrow the L2, 94.7 / 96.5: not.  Open:
//   32 x 1024 24.4 / 26.6.
//   257 to 512, masks as values (what they hide is not known here), causal, open, window,
//   hidden: head 64, 36 x 500 15.5 15.2 13.6 4.5 / 12.1 14.0 10.9 4.3, 32 x 1024 20.8 20.5 14.3 4.5 / 16.8
//   19.9 12.0 4.5, 9 x 2048 26.8 28.2 15.0 7.0 / 23.4 29.1 14.1 6.0, 16 x 2048 28.1 30.4 15.7 7.3 / 24.9
//   31.1 13.4 6.0; up to 768 24 x 2000 35.5 46.0 18.3 6.3 / 28.0 43.1 16.7 6.8, 64 x 700 17.7 23.3 15.7
//   4.9 / 15.8 21.6 13.8 4.8; head 128, 16 x 1500 33.1 35.5 18.9 6.3 / 25.9 34.9 16.4 5.6, 16 x 2048 39.6
//   46.9 22.6 8.6 / 33.0 47.1 19.4 7.6, 15 x 1622 35.3 37.6 19.4 6.5 / 30.8 37.5 18.0 5.7; with fewer
//   steps 32 x 1024 27.6 27.3 - 5.0 / 24.1 30.0 - 6.4: not; nor where the keys outgrow the L2.
static bool halved_is_faster(const PrefillParams &p, int head, int mode)
{
    const int64_t tiles = (int64_t)p.batch * p.n_slabs * p.n_q_tiles;
    constexpr int64_t kCUs = 8 * kCUsPerXCD;
    const int64_t n_wg = tiles * ((p.q_tile + kQRows / 2 - 1) / (kQRows / 2));
    const bool three = head == 64 && mode != NNTILE_HIP_MASK_NONE && n_wg <= 3 * kCUs
        && (tiles % 8 == 0 || (mode == NNTILE_HIP_MASK_CAUSAL && p.k_seq >= 64 * kKeys));
    if(!three && tiles * ((p.q_tile + kQRows - 1) / kQRows) > kCUs)
    {
        return false;
    }
    const int64_t steps = key_steps(p);
    const bool rule = mode == NNTILE_HIP_MASK_CAUSAL || mode == NNTILE_HIP_MASK_NONE;
    if(rule && p.q_seq != p.k_seq && steps < kHalvedSteps)
    {
        return false;
    }
    switch(mode)
    {
        case NNTILE_HIP_MASK_CAUSAL:
            // (beyond 256 workgroups where the rule hides enough to make long and short
            // ones: 64 heads, 333 queries behind 1500 keys 33.9 / 36.8)
            return n_wg <= kCUs || (p.q_pos0 + p.causal_offset - p.k_pos0 < p.k_seq / 2
                    && (head == 64 ? 2 : 1) * keys_on_xcd(p, head).fit >= steps);
        case NNTILE_HIP_MASK_NONE:
            return n_wg <= kCUs && (steps < 2 * kTouchSteps || 2 * keys_on_xcd(p, head).fit >= steps);
        default:
            return n_wg <= kCUs || (steps >= kTouchStepsMask ? keys_on_xcd(p, head).fit >= steps : head == 64);
    }
}

// Which lines of K and V the workgroups of a launch touch before they begin.
static void set_touch(PrefillParams &p, int head, int mode, int64_t n_wg)
{
    const int64_t steps = key_steps(p);
    const bool rule = mode == NNTILE_HIP_MASK_CAUSAL || mode == NNTILE_HIP_MASK_NONE;
    if(steps < (rule || head == 64 || n_wg <= 8 * kCUsPerXCD ? kTouchSteps : kTouchStepsMask))
    {
        return;
    }
    const KeysOnXCD keys = keys_on_xcd(p, head);
    if(3 * keys.fit >= steps)
    {
        p.touch_group = keys.group;
        p.touch_steps = (int)std::min(steps, keys.fit);
    }
}

// Host launcher shared by the tile and grid entry points.  p must be fully
// filled except for the block counts and the remap flag.  scan_scratch: device
// memory the call may use for a scan of an explicit mask (may be null).
template<typename T>
int launch_prefill_16bit(hipStream_t stream, PrefillParams &p, int head,
        int mode, void *scan_scratch, size_t scan_scratch_bytes)
{
    // 256-query workgroups (eight wavefronts, one workgroup a CU): when asked
    // for (p.form from 8 on), and by themselves where they measured faster - head
    // 128, whole 256-query blocks, and enough of them that every CU gets two
    // under a causal mask (one workgroup a CU has nobody to share the CU with
    // while it starts and ends, and a causal launch of one round is set by its
    // longest workgroup), or a whole number of rounds without a mask.
    // p.form == 1 keeps the 128-query form.
    const bool can_wide = (head == 64 || head == 128)
        && (mode == NNTILE_HIP_MASK_NONE || mode == NNTILE_HIP_MASK_CAUSAL);
    bool wide = can_wide && p.form >= 8;
    if(can_wide && p.form == 0 && head == 128 && (p.q_tile % 256 == 0 || p.n_q_tiles == 1))
    {
        const int64_t n_w = (int64_t)p.batch * p.n_slabs * p.n_q_tiles * ((p.q_tile + 255) / 256);
        wide = mode == NNTILE_HIP_MASK_CAUSAL ? n_w >= 512
            : (n_w >= 256 && (n_w % 256 == 0 || n_w >= 1024));
    }
    const bool can_halve = (head == 64 || head == 128) && !wide;
    const bool halved = can_halve
        && (p.form == 3 || (p.form == 0 && halved_is_faster(p, head, mode)));
    const int q_rows = wide ? 256 : halved ? kQRows / 2 : kQRows;
    p.q_blocks_per_tile = (int)((p.q_tile + q_rows - 1) / q_rows);
    p.k_blocks_per_tile = (int)((p.k_tile + kKeys - 1) / kKeys);
    const int64_t batch_all = (int64_t)p.batch * p.n_slabs;
    const int64_t n_wg = batch_all * p.n_q_tiles * p.q_blocks_per_tile;
    if(n_wg <= 0 || n_wg > 0x7fffffff)
    {
        return NNTILE_HIP_EINVAL;
    }
    // Two groups of four wavefronts per workgroup, each taking every second
    // key step (p.form == 2, or by itself): when the launch has at most one
    // 128-query workgroup per CU, so that a CU would otherwise hold one wavefront
    // per SIMD, is none of those that halve the steps, and has enough key steps to share.
    // Without a mask: as fast at 1024 keys, 12-20 % less on longer rows (head 64: 3-8 % less at
    // 1024 keys); shorter rows lose by it (head 128, 36 x 512 14.1 / 15.9, 4 x 300 11.0 / 12.6; head
    // 64 10.7 / 11.2, 8.7 / 9.3).  Masks
    // given as values, head 128: 1024 keys 25.3 us with four wavefronts, 28.6 with two
    // groups (32 heads), 4096 keys 7-11 % less; head 64: 2048 keys 28.8 / 28.2 (16 heads).
    const bool can_split = can_halve && !halved;
    const bool explicit_mask = mode == NNTILE_HIP_MASK_ADDITIVE || mode == NNTILE_HIP_MASK_BOOL;
    // (head 64 under such a mask comes here with 24 steps and more)
    const bool key_split = can_split && (p.form == 2
            || (p.form == 0 && n_wg <= 8 * (int64_t)kCUsPerXCD
                && p.k_seq >= (explicit_mask ? (head == 64 ? 24 : 32) : head == 64 ? 12 : 16) * kKeys));
    p.touch_steps = 0;
    if(halved)
    {
        set_touch(p, head, mode, n_wg);
    }
    p.mask_bits = nullptr;
    const int scan_rc = scan_mask_once<T>(stream, p, mode, halved, scan_scratch, scan_scratch_bytes);
    if(scan_rc != NNTILE_HIP_OK)
    {
        return scan_rc;
    }
    p.xcd_remap = (batch_all % 8 == 0) ? 1 : 0;
    // (the scanning workgroups come first; their number is a multiple of 8, so
    // the attention workgroups keep their places in the round of the XCDs)
    const dim3 grid((unsigned)(n_wg + p.n_scan_wgs));
    switch(head)
    {
        case 32:
            return launch_mode<T, 32>(stream, p, mode, grid, false, false, false);
        case 64:
            return launch_mode<T, 64>(stream, p, mode, grid, wide, key_split, halved);
        case 128:
            return launch_mode<T, 128>(stream, p, mode, grid, wide, key_split, halved);
        default:
            return NNTILE_HIP_EUNSUPPORTED;
    }
}

// One tile against a long key axis, the keys in p.n_parts ranges (set by the
// caller from prefill_parts, with p.part_*; p.kv_rows must be given).
template<typename T>
int launch_prefill_16bit_parts(hipStream_t stream, PrefillParams &p, int head, int mode)
{
    p.q_blocks_per_tile = (int)((p.q_tile + kQRows - 1) / kQRows);
    p.k_blocks_per_tile = (int)((p.k_tile + kKeys - 1) / kKeys);
    p.mask_bits = nullptr;
    p.n_scan_wgs = 0;
    p.touch_steps = 0;
    p.xcd_remap = (p.batch % 8 == 0) ? 1 : 0;
    const dim3 grid((unsigned)((int64_t)p.batch * p.q_blocks_per_tile * p.n_parts));
    const bool causal = mode == NNTILE_HIP_MASK_CAUSAL;
    auto launch = [&](auto kernel) -> int
    {
        hipLaunchKernelGGL(kernel, grid, dim3(512), 0, stream, p);
        return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
    };
    switch(head)
    {
        case 64:
            return causal
                ? launch(sdpa_prefill_16bit_kernel<T, 64, NNTILE_HIP_MASK_CAUSAL, 8, 2, true>)
                : launch(sdpa_prefill_16bit_kernel<T, 64, NNTILE_HIP_MASK_NONE, 8, 2, true>);
        case 128:
            return causal
                ? launch(sdpa_prefill_16bit_kernel<T, 128, NNTILE_HIP_MASK_CAUSAL, 8, 2, true>)
                : launch(sdpa_prefill_16bit_kernel<T, 128, NNTILE_HIP_MASK_NONE, 8, 2, true>);
        default:
            return NNTILE_HIP_EUNSUPPORTED;
    }
}

template int launch_prefill_16bit_parts<Bf16>(hipStream_t, PrefillParams &, int, int);
template int launch_prefill_16bit_parts<Fp16>(hipStream_t, PrefillParams &, int, int);
template int launch_prefill_16bit<Bf16>(hipStream_t, PrefillParams &, int, int, void *, size_t);
template int launch_prefill_16bit<Fp16>(hipStream_t, PrefillParams &, int, int, void *, size_t);

} // namespace nntile_hip
