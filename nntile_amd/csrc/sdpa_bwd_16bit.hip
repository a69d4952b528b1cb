// Scaled dot-product attention backward for 16-bit tiles on gfx950, in the
// flash form: the forward output A and the logsumexp are inputs, the
// probabilities are recomputed from them,
//
//   P[q,k]  = exp(scale q.k + mask[q,k] - lse[q])        D[q] = dA[q,:] . A[q,:]
//   dP[q,k] = dA[q,:] . V[k,:]                           dS   = P (dP - D)
//   dV[k,:] += sum_q P[q,k] dA[q,:]      dQ[q,:] += scale sum_k dS[q,k] K[k,:]
//   dK[k,:] += scale sum_q dS[q,k] Q[q,:]
//
// (include/nntile/kernel/flash_sdpa_bwd_cudnn/cuda.hh:44-68 is the interface
// this replaces; tests/kernel/flash_sdpa_bwd_cudnn.cc:174-262 the arithmetic).
// A small launch writes D (and looks over a mask given as values); then ONE
// launch computes the three gradients, each
// by its own workgroups (no atomics, results independent of timing):
//
//  * sdpa_bwd_dq_body: a workgroup owns 128 queries (a wavefront 32, a lane
//    one query) and walks the keys in steps of 64, as the forward kernel does:
//    S^T = K Q^T and dP^T = V dA^T with Q and dA fragments in registers and K, V
//    rows from LDS; dS^T packed to 16 bits is the B operand of
//    dQ^T += K^T dS^T, whose A operand comes through the transposing LDS read.
//  * sdpa_bwd_dkv_body<PART>: a workgroup owns 128 keys (a lane one key) and
//    walks the queries of every head of its group in steps of 64: S = Q K^T
//    and dP = dA V^T with K and V fragments in registers and Q, dA rows from
//    LDS; dV^T += dA^T P or dK^T += Q^T dS (PART) through transposing reads of
//    the same two LDS tiles.
//
// K, V, Q, dA steps go from global memory straight into LDS, double buffered;
// 16-byte chunk c of row r of a step sits at chunk position c ^ swz(r)
// (BwdTile::swz), which keeps both the row reads and the transposing reads
// free of bank conflicts.
#include <type_traits>
#include <utility>

#include "sdpa_common.hpp"

namespace nntile_hip
{

// Developer build (-DNNTILE_BWD_TRACE): shader-clock cycles that the first
// wavefront of every key-owning workgroup spends in each phase of its steps,
// summed over the steps; read back with nntile_hip_debug_bwd_trace.
#ifdef NNTILE_BWD_TRACE
__device__ unsigned long long bwd_trace[8 * 4096];
__device__ unsigned long long bwd_wall[4 * 4096];
#define BWD_WALL(i, part) do { if(threadIdx.x == 0 && blockIdx.x < 4096) { \
        bwd_wall[4 * blockIdx.x + (i)] = wall_clock64(); bwd_wall[4 * blockIdx.x + 2] = (part); } } while(0)
#define BWD_WALL_AT(i) do { if(threadIdx.x == 0 && blockIdx.x < 4096) { \
        bwd_wall[4 * blockIdx.x + (i)] = wall_clock64(); } } while(0)
#define BWD_TRACE_DECL unsigned long long bt_sum[7] = {0, 0, 0, 0, 0, 0, 0}, bt_last = 0; int bt_steps = 0;
#define BWD_TRACE_START() do { bt_last = clock64(); } while(0)
#define BWD_TRACE_MARK(i) do { const unsigned long long now_ = clock64(); bt_sum[i] += now_ - bt_last; \
        bt_last = now_; } while(0)
#define BWD_TRACE_STEP() do { bt_steps += 1; } while(0)
#define BWD_TRACE_FLUSH(part) do { if(threadIdx.x == 0 && blockIdx.x < 4096) { \
        for(int i_ = 0; i_ < 6; ++i_) { bwd_trace[8 * blockIdx.x + i_] = bt_sum[i_]; } \
        bwd_trace[8 * blockIdx.x + 6] = (unsigned long long)bt_steps; \
        bwd_trace[8 * blockIdx.x + 7] = (unsigned long long)(part); } } while(0)
}
extern "C" int nntile_hip_debug_bwd_wall(unsigned long long *host)
{
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(nntile_hip::bwd_wall), sizeof(nntile_hip::bwd_wall));
}
extern "C" int nntile_hip_debug_bwd_trace(unsigned long long *host)
{
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(nntile_hip::bwd_trace), sizeof(nntile_hip::bwd_trace));
}
namespace nntile_hip
{
#else
#define BWD_TRACE_DECL
#define BWD_TRACE_START()
#define BWD_TRACE_MARK(i)
#define BWD_TRACE_STEP()
#define BWD_TRACE_FLUSH(part)
#define BWD_WALL(i, part)
#define BWD_WALL_AT(i)
#endif


// 1: a step's two query (key) blocks overlap - the matrix products of one
// beside the vector work of the other; 0: one block after the other
#ifndef NNTILE_BWD_PIPE
#define NNTILE_BWD_PIPE 1
#endif
#ifndef NNTILE_BWD_PIPE_DQ
#define NNTILE_BWD_PIPE_DQ 1        // the same in the dQ workgroups
#endif
#ifndef NNTILE_BWD_AHEAD
#define NNTILE_BWD_AHEAD 2          // LDS operands are read this many MFMAs early, head 128
#endif
#ifndef NNTILE_BWD_AHEAD_NARROW
#define NNTILE_BWD_AHEAD_NARROW 4   // and at head 32 and 64, whose bodies have the registers
#endif
#ifndef NNTILE_BWD_AHEAD_WIDE
#define NNTILE_BWD_AHEAD_WIDE 2     // the same where a workgroup holds both gradients at head 128
#endif
// Where the tile loads of the next step are issued: 0 = all at the start of
// the step, 1 = between the MFMAs of the step's first half, 2 = of the whole
#ifndef NNTILE_BWD_SPREAD
#define NNTILE_BWD_SPREAD 2
#endif
#ifndef NNTILE_BWD_SWIZZLE_ROTATED
#define NNTILE_BWD_SWIZZLE_ROTATED 1
#endif
constexpr int kBwdRows = 128;       // queries (dQ workgroups) / keys (dK, dV workgroups) per workgroup
constexpr int kBwdStep = 64;        // rows of the other axis per step
constexpr int kBwdThreads = 256;
template<int HEAD> constexpr int kBwdAhead = HEAD > 64 ? NNTILE_BWD_AHEAD : NNTILE_BWD_AHEAD_NARROW;

__device__ __forceinline__ u32x2 bwd_lds_read_tr16(const char *lds_ptr)
{
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(lds_ptr));
    return __builtin_bit_cast(u32x2, v);
}

// What the three kinds of workgroup share: the geometry of a 64-row step in LDS.
template<int HEAD>
struct BwdTile
{
    static constexpr int KSTEPS = HEAD / 16;       // MFMA steps along head
    static constexpr int DBLOCKS = HEAD / 32;      // 32-row blocks of a transposed gradient
    static constexpr int RB = HEAD * 2;            // bytes per row
    static constexpr int CPR = HEAD / 8;           // 16-byte chunks per row
    static constexpr int RPL = 16 / CPR;           // rows per 256-byte line of LDS banks
    static constexpr int ROWS_PER_LOAD = 1024 / RB;
    static constexpr int LOADS = kBwdStep / ROWS_PER_LOAD;
    static constexpr int LOADS_PER_WAVE = LOADS / 4;
    static constexpr int BYTES = kBwdStep * RB;
    static_assert(LOADS_PER_WAVE >= 1, "head size does not fit this tiling");

    // Chunk c of row r sits at chunk position c ^ swz(r).  Every tile is read
    // both ways: 16 lanes read the same chunk of 16 consecutive rows (they
    // need 16 different positions: swz must be one-to-one on 16 rows), and 32
    // lanes of a transposing read take 4 neighbouring chunks of 4 consecutive
    // rows (the 4 rows need different groups of 4 positions: the low bits of
    // the line number must land in the top bits).  Both hold for the line
    // number (r / RPL) % CPR rotated right by log2(CPR) - 2 bits.
    static __device__ __forceinline__ int swz(int r)
    {
        constexpr int ROT = CPR == 16 ? 2 : (CPR == 8 ? 1 : 0);
        constexpr int BITS = CPR == 16 ? 4 : (CPR == 8 ? 3 : 2);
        const int line = (r / RPL) % CPR;
#if NNTILE_BWD_SWIZZLE_ROTATED
        return ((line >> ROT) | (line << (BITS - ROT))) & (CPR - 1);
#else
        return line;
#endif
    }
};

// The registers of a 32x32 accumulator tile of lane (col, half): register r is
// row 8*(r/4) + 4*half + r%4 of the tile, column col.
// Workgroup number -> (batch entry, block along the sequence).  Workgroups
// go to the 8 XCDs round robin: the entries of the batch are dealt so that
// all blocks of one entry run on one XCD and share its L2, and the blocks are
// taken in the order longest first (`last_first`: from the last block down).
__device__ __forceinline__ void map_workgroup(unsigned wg, int entries, int blocks,
        bool last_first, int &entry, int &block)
{
    int i;
    if((entries & 7) == 0)
    {
        const int per_xcd = entries >> 3;
        i = (int)(wg >> 3);
        entry = (int)(wg & 7u) * per_xcd + i % per_xcd;
        i /= per_xcd;
    }
    else
    {
        entry = (int)(wg % (unsigned)entries);
        i = (int)(wg / (unsigned)entries);
    }
    // (the same for every lane: into scalar registers, whatever the divisions
    // were computed with)
    entry = __builtin_amdgcn_readfirstlane(entry);
    block = __builtin_amdgcn_readfirstlane(last_first ? blocks - 1 - i : i);
}

// The lane's index within its wavefront, asked of the hardware where it is
// needed again after a long loop (the thread index the kernel started with
// would have to sit in a register all the way through, and at head 128 there
// is none to spare).  Does not depend on which lanes are active.
__device__ __forceinline__ int lane_index_again()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// base ^ BITS, in assembly text: the compiler would make all the places that
// differ by a constant once, before the loop, and spill them.
template<int BITS>
__device__ __forceinline__ uint32_t flip_bits(uint32_t base)
{
    uint32_t r;
    asm volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(BITS), "v"(base));
    return r;
}

// f(0), f(1), .. f(N-1), each index a compile-time constant
template<typename F, int... I>
__device__ __forceinline__ void each_slot(F f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}

__device__ __forceinline__ int tile_row(int r, int half)
{
    return 8 * (r >> 2) + 4 * half + (r & 3);
}

// ---------------------------------------------------------------------------------
// What the gradient launch needs first, in one launch of its own (the row dots
// tile by tile and the classes of the mask blocks apart were up to nine
// launches; each costs the stream 2 to 4 us):
//
//  * the row dots D[b][q] = dA[b][q][:] . A[b][q][:] in fp32: 16-byte loads,
//    HEAD/8 lanes a row, kRowdotRows rows per lane in flight, summed across
//    those lanes;
//  * for a mask given as values the class of every 64 x 64 block (the
//    reference hands the kernel a materialised tile even where it is causal,
//    src/tile/flash_sdpa_bwd_cudnn.cc), so that the gradient bodies skip the
//    steps whose blocks hide everything - without fetching them - and read mask
//    values only where they must: not in blocks that mask nothing, and not in
//    blocks that hold exactly what the rule `key <= query` (rows and columns
//    of this tile) makes of them - the diagonal blocks of a causal tile.
//
// Class bits of a block: some value is visible; some value is not "open" (+0 /
// true); some value is not what the rule says.
constexpr int kMaskVisible = 1, kMaskMasked = 2, kMaskOffRule = 4;
constexpr int kRowdotRows = 2;

struct BwdPreludeParams
{
    int64_t q_seq, q_tile, mask_ld;
    float *D;
    const void *mask;
    uint8_t *table;
    int32_t k_seq, class_ld;        // (masks: one tile of each axis)
    int32_t batch, n_q_tiles;       // slab s's tiles at [s*n_q_tiles + t] of the tables
    int32_t n_class_wgs, wgs_per_tile;
    const void *dA[kBwdMaxTiles];
    const void *A[kBwdMaxTiles];
};

// Class bits of the thread's 16 of a block's 64 x 64 values: row `row`, from column col0 on
// (threads 4 * r + i: row r of the block, columns 16 * i ..; none past the end).
template<typename T, int MODE>
__device__ __forceinline__ uint32_t bwd_piece_class(const void *mask, int64_t mask_ld, int q_seq,
        int k_seq, int row, int col0)
{
    constexpr int ES = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 2 : 1;
    constexpr int PER_WORD = 4 / ES;
    constexpr uint32_t OPEN = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 0u : 0x01010101u;
    constexpr uint32_t HIDDEN = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? T::kNegInfPair : 0u;
    typedef u32x4 __attribute__((aligned(1))) u32x4_any;
    uint32_t seen = 0u;
    if(row < q_seq && col0 < k_seq)
    {
        const char *src = static_cast<const char *>(mask) + ((int64_t)row * mask_ld + col0) * ES;
        const int n_vis = row - col0 + 1;       // columns of this thread that the rule shows
        if(col0 + 16 <= k_seq)
        {
            // the thread's 16 values as 16-byte loads of any alignment
            u32x4 v[ES];
#pragma unroll
            for(int i = 0; i < ES; ++i)
            {
                v[i] = *reinterpret_cast<const u32x4_any *>(src + 16 * i);
            }
            uint32_t masked = 0u, visible = 0u, off = 0u;
#pragma unroll
            for(int w = 0; w < 4 * ES; ++w)
            {
                const uint32_t x = v[w / 4][w % 4];
                masked |= x ^ OPEN;
                visible |= x ^ HIDDEN;
                // elements PER_WORD*w ..: the first n of them are shown
                const int n = min(max(n_vis - PER_WORD * w, 0), PER_WORD);
                const uint32_t low = n == PER_WORD ? ~0u : (1u << (8 * ES * n)) - 1u;
                off |= x ^ ((OPEN & low) | (HIDDEN & ~low));
            }
            seen = (visible != 0u ? kMaskVisible : 0) | (masked != 0u ? kMaskMasked : 0)
                | (off != 0u ? kMaskOffRule : 0);
        }
        else
        {
            for(int e = 0; e < k_seq - col0; ++e)
            {
                bool open, hidden;
                if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                {
                    const uint16_t x = reinterpret_cast<const uint16_t *>(src)[e];
                    open = x == 0;              // anything but +0 changes the score
                    hidden = x == (uint16_t)T::kNegInfPair;
                }
                else
                {
                    open = reinterpret_cast<const uint8_t *>(src)[e] == 1;
                    hidden = reinterpret_cast<const uint8_t *>(src)[e] == 0;
                }
                seen |= (!hidden ? kMaskVisible : 0) | (!open ? kMaskMasked : 0)
                    | ((e < n_vis ? !open : !hidden) ? kMaskOffRule : 0);
            }
        }
    }
    return seen;
}

template<typename T, int MODE>
__device__ __forceinline__ void bwd_mask_class(const BwdPreludeParams &p, int wg)
{
    const uint32_t seen = bwd_piece_class<T, MODE>(p.mask, p.mask_ld, (int)p.q_seq, p.k_seq,
            wg / p.class_ld * kBwdStep + (int)threadIdx.x / 4,
            wg % p.class_ld * kBwdStep + ((int)threadIdx.x % 4) * 16);
    uint32_t all = 0u;
#pragma unroll
    for(int b = 0; b < 3; ++b)
    {
        all |= __syncthreads_or((int)(seen & (1u << b))) != 0 ? (1u << b) : 0u;
    }
    if(threadIdx.x == 0)
    {
        p.table[wg] = (uint8_t)all;
    }
}

// Eight products of a row dot, one after the other.  (The products are exact in 32 bits.
// Nothing may be contracted: in fp16 the compiler takes a two-way dot product where it finds
// the pattern, which rounds otherwise, and the same row must give the same bits wherever
// its dot is taken.)
template<typename T>
__device__ __forceinline__ float bwd_dot8(const u32x4 &g, const u32x4 &a)
{
#pragma clang fp contract(off)
    float d = 0.0f;
#pragma unroll
    for(int e = 0; e < 4; ++e)
    {
        d = __builtin_fmaf(T::to_float((uint16_t)(g[e] & 0xffffu)),
                T::to_float((uint16_t)(a[e] & 0xffffu)), d);
        d = __builtin_fmaf(T::to_float((uint16_t)(g[e] >> 16)), T::to_float((uint16_t)(a[e] >> 16)), d);
    }
    return d;
}

template<typename T, int HEAD, int MODE>
__global__ __launch_bounds__(256)
void sdpa_bwd_prelude_kernel(const BwdPreludeParams p)
{
    if constexpr(MODE == NNTILE_HIP_MASK_ADDITIVE || MODE == NNTILE_HIP_MASK_BOOL)
    {
        if((int)blockIdx.x < p.n_class_wgs)
        {
            bwd_mask_class<T, MODE>(p, (int)blockIdx.x);
            return;
        }
    }
    constexpr int LANES = HEAD / 8;             // lanes per row: 16, 8 or 4
    constexpr int ROWS = 256 / LANES;           // rows one load of the workgroup covers
    const int wg = (int)blockIdx.x - p.n_class_wgs;
    const int tile = wg / p.wgs_per_tile;
    const int64_t t0 = (int64_t)(tile % p.n_q_tiles) * p.q_tile;
    const int64_t rows = (int64_t)p.batch * min(p.q_tile, p.q_seq - t0);
    const int64_t row0 = (int64_t)(wg % p.wgs_per_tile) * (ROWS * kRowdotRows)
        + (int)threadIdx.x / LANES;
    const int part = (int)(threadIdx.x % LANES);
    const uint16_t *dA = static_cast<const uint16_t *>(p.dA[tile]) + part * 8;
    const uint16_t *A = static_cast<const uint16_t *>(p.A[tile]) + part * 8;
    float *D = p.D + (int64_t)(tile / p.n_q_tiles) * p.q_seq * p.batch + (int64_t)p.batch * t0;
    u32x4 g[kRowdotRows], a[kRowdotRows];
#pragma unroll
    for(int i = 0; i < kRowdotRows; ++i)
    {
        // (rows past the end read the last one)
        const int64_t row = min(row0 + i * ROWS, rows - 1);
        g[i] = *reinterpret_cast<const u32x4 *>(dA + row * HEAD);
        a[i] = *reinterpret_cast<const u32x4 *>(A + row * HEAD);
    }
#pragma unroll
    for(int i = 0; i < kRowdotRows; ++i)
    {
        float d = bwd_dot8<T>(g[i], a[i]);
#pragma unroll
        for(int o = LANES / 2; o >= 1; o >>= 1)
        {
            d += __shfl_xor(d, o, 64);
        }
        if(row0 + i * ROWS < rows && part == 0)
        {
            D[row0 + i * ROWS] = d;
        }
    }
}

// ---- without the launch in front ---------------------------------------------------
// Walks of up to two blocks (OWN below): every workgroup finds out for itself what
// it needs, with the arithmetic of the launch in front and so the same bits: the row dots of
// its queries, the classes of the blocks that it meets.  A launch costs about 2.5 us before the
// next one starts, the same work inside the workgroups the latency of one round of loads, and
// more with each 128 rows that a key block's workgroup needs the dots of.  Measured (us, with the
// launch / without): head 64, causal by rule, 4 x 64 7.2 / 5.3, 12 x 128 8.3 / 6.3, 64 x 128 10.0 / 7.6;
// masks, 12 x 64 8.7 / 7.2, 40 x 128 10.0 / 9.0; head 128, causal by rule, 32 x 60 9.8 / 7.7, 64 x 128
// 14.3 / 11.9; masks, 12 x 64 10.9 / 9.9, 4 x 128 11.6 / 11.7.  Longer walks lose (a variant that
// took them, against its own form with the launch): masks, 8 x 200 of head 64 11.6 / 14.5, head
// 128 14.9 / 19.0; by rule, 32 x 60 in groups of 4 10.4 / 11.7, 12 x 200 of head 128 12.9 / 14.1, and
// of head 64 10.2 / 9.5 but 12 x 400 12.7 / 13.0.
constexpr int kBwdOwnRows = 128;            // queries of a walk, all heads of a group
constexpr int kBwdOwnSteps = kBwdOwnRows / kBwdStep;

// Row dots of `rows` rows, q_seq of each head of a group, by 256 threads, into out.  dA, A:
// the first; head_gap: elements between the rows of one head and those of the next.
// (All heads in one run: a loop over the heads waits for memory once for each, and a
// group of many heads has few rows of one.  With the launch in front / a loop / now, us, bf16, no
// mask: head 64, 2 groups of 128 heads of a row 115 / 189 / 88, 4 of 32 x 4 30 / 50 / 24, 8 of 16 x 8
// 18.7 / 27 / 14.7, 2 of 8 x 16 12.8 / 15.5 / 9.4, 16 of 4 x 32 10.0 / 10.1 / 7.3; head 128, 2 of 128 x
// 1 151 / 231 / 116, 8 of 16 x 8 26 / 35 / 21.)
template<typename T, int HEAD>
__device__ __forceinline__ void bwd_own_row_dots(const uint16_t *dA, const uint16_t *A, int rows,
        int q_seq, int64_t head_gap, float *out)
{
    constexpr int LANES = HEAD / 8, ROWS = 256 / LANES, N = 4;
    const int part = (int)threadIdx.x % LANES, row0 = (int)threadIdx.x / LANES;
    for(int base = 0; base < rows; base += N * ROWS)
    {
        u32x4 g[N], a[N];
#pragma unroll
        for(int i = 0; i < N; ++i)
        {
            const int row = min(base + i * ROWS + row0, rows - 1);
            const int64_t at = (rows > q_seq ? row / q_seq * head_gap : 0) + row * HEAD + part * 8;
            g[i] = *reinterpret_cast<const u32x4 *>(dA + at);
            a[i] = *reinterpret_cast<const u32x4 *>(A + at);
        }
#pragma unroll
        for(int i = 0; i < N; ++i)
        {
            float d = bwd_dot8<T>(g[i], a[i]);
#pragma unroll
            for(int o = LANES / 2; o >= 1; o >>= 1)
            {
                d += __shfl_xor(d, o, 64);
            }
            if(base + i * ROWS + row0 < rows && part == 0)
            {
                out[base + i * ROWS + row0] = d;
            }
        }
    }
}

// Classes of the blocks own0 x [first, last) (by_row: the owned block is one of queries),
// three bits each, in the order of the walk.  word: one word of LDS, zero before.
template<typename T, int MODE>
__device__ __forceinline__ uint32_t bwd_own_classes(const BwdParams &p, int own0, int first, int last,
        bool by_row, uint32_t *word)
{
    const int r = (int)threadIdx.x / 4, c = ((int)threadIdx.x % 4) * 16;
    uint32_t seen[kBwdOwnSteps];
#pragma unroll
    for(int i = 0; i < kBwdOwnSteps; ++i)
    {
        const int g = first + i;
        seen[i] = g < last ? bwd_piece_class<T, MODE>(p.mask, p.mask_ld, (int)p.q_seq, (int)p.k_seq,
                (by_row ? own0 : g) * kBwdStep + r, (by_row ? g : own0) * kBwdStep + c) : 0u;
    }
    uint32_t all = 0u;
#pragma unroll
    for(int i = 0; i < kBwdOwnSteps; ++i)
    {
#pragma unroll
        for(int b = 0; b < 3; ++b)
        {
            all |= __builtin_amdgcn_ballot_w64((seen[i] & (1u << b)) != 0u) != 0ull ? 1u << (3 * i + b) : 0u;
        }
    }
    if(threadIdx.x % 64 == 0)
    {
        atomicOr(word, all);
    }
    __syncthreads();
    return *word;
}

// The steps a workgroup takes, as a bit set (up to 64 of them; longer walks
// take every step), the subset in which nothing is masked and the subset in
// which the mask is the rule `key <= query`.
struct StepSet
{
    unsigned long long active, open, rule;
    bool use_bits;
    int first, last;        // [first, last): the walk without the table

    __device__ __forceinline__ int begin() const
    {
        if(!use_bits)
        {
            return first < last ? first : -1;
        }
        return active != 0ull ? __builtin_ctzll(active) : -1;
    }
    __device__ __forceinline__ int next(int g) const
    {
        if(!use_bits)
        {
            return g + 1 < last ? g + 1 : -1;
        }
        const unsigned long long rest = g >= 63 ? 0ull : (active >> (g + 1)) << (g + 1);
        return rest != 0ull ? __builtin_ctzll(rest) : -1;
    }
    __device__ __forceinline__ bool is_open(int g) const
    {
        return use_bits && ((open >> g) & 1ull) != 0ull;
    }
    __device__ __forceinline__ bool is_rule(int g) const
    {
        return use_bits && ((rule >> g) & 1ull) != 0ull;
    }
};

// Step set of a workgroup that owns the blocks [own0, own0 + n_own) of one axis
// and walks the blocks [first, last) of the other.  by_row: the owned blocks
// are query blocks (rows of the table).
__device__ __forceinline__ StepSet make_step_set(const BwdParams &p, bool explicit_mask,
        int own0, int n_own, int first, int last, bool by_row, bool own = false, uint32_t own_bits = 0u)
{
    StepSet s;
    s.first = first;
    s.last = last;
    s.use_bits = explicit_mask && (own || p.mask_class != nullptr) && last <= 64;
    s.active = 0ull;
    s.open = 0ull;
    s.rule = 0ull;
    if(s.use_bits)
    {
        // lane g looks at step g; the ballots make the two sets (every
        // wavefront computes the same)
        const int g = (int)(threadIdx.x & 63);
        const bool in_walk = g >= first && g < last;
        int c = 0;
        if(own)
        {
            c = in_walk ? (int)(own_bits >> (3 * min(g - first, kBwdOwnSteps))) & 7 : 0;
        }
        for(int o = 0; !own && o < n_own; ++o)
        {
            const int idx = by_row ? (own0 + o) * p.class_ld + g : g * p.class_ld + own0 + o;
            c |= in_walk ? p.mask_class[idx] : 0;
        }
        s.active = __builtin_amdgcn_ballot_w64(in_walk && (c & kMaskVisible) != 0);
        s.open = __builtin_amdgcn_ballot_w64(in_walk && (c & kMaskMasked) == 0);
        s.rule = __builtin_amdgcn_ballot_w64(in_walk && (c & kMaskOffRule) == 0);
    }
    return s;
}

// A wavefront's 32 rows of a gradient (accumulators acc, transposed: register r
// of block db is head value db*32 + tile_row(r, half) of row lane % 32), times
// factor, to memory through LDS - so that they leave, and what they are added
// to arrives, as whole rows, 16 bytes a lane, instead of 8-byte pieces 2*HEAD
// bytes apart.  xch: 32 rows of LDS of the wavefront's own; base: the first
// row; n_ok: rows that exist (may be none or more than 32).
// KH == 2: half of each row, the blocks in front of acc; base: where that half begins.
template<typename T, int HEAD, int KH = 1>
__device__ __forceinline__ void bwd_store_rows(char *xch, char *base, int n_ok,
        const f32x16 (&acc)[HEAD / 32], float factor, bool add)
{
    typedef BwdTile<HEAD> G;
    constexpr int STRIDE = G::RB, RB = G::RB / KH, CPR = G::CPR / KH, RPI = 1024 / RB, N = 32 / RPI;
    if(n_ok <= 0)
    {
        return;
    }
    const int lane = lane_index_again();
    const int st_row = lane / CPR, st_c = lane % CPR;
    if(add)
    {
        u32x4 old[N];
#pragma unroll
        for(int i = 0; i < N; ++i)
        {
            old[i] = *reinterpret_cast<const u32x4 *>(base
                    + (int64_t)min(i * RPI + st_row, n_ok - 1) * STRIDE + st_c * 16);
        }
#pragma unroll
        for(int i = 0; i < N; ++i)
        {
            const int r = i * RPI + st_row;
            *reinterpret_cast<u32x4 *>(xch + r * RB + (st_c ^ (r % CPR)) * 16) = old[i];
        }
    }
    const int col = lane & 31, half = lane >> 5;
#pragma unroll
    for(int db = 0; db < G::DBLOCKS / KH; ++db)
    {
#pragma unroll
        for(int rg = 0; rg < 4; ++rg)
        {
            u32x2 *at = reinterpret_cast<u32x2 *>(xch + col * RB
                    + ((db * 4 + rg) ^ (col % CPR)) * 16 + 8 * half);
            float v[4];
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                v[e] = acc[db][4 * rg + e] * factor;
            }
            if(add)
            {
                const u32x2 old = *at;
                v[0] += T::to_float((uint16_t)(old[0] & 0xffffu));
                v[1] += T::to_float((uint16_t)(old[0] >> 16));
                v[2] += T::to_float((uint16_t)(old[1] & 0xffffu));
                v[3] += T::to_float((uint16_t)(old[1] >> 16));
            }
            *at = u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
        }
    }
#pragma unroll
    for(int i = 0; i < N; ++i)
    {
        const int r = i * RPI + st_row;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(xch + r * RB + (st_c ^ (r % CPR)) * 16);
        if(r < n_ok)
        {
            *reinterpret_cast<u32x4 *>(base + (int64_t)r * STRIDE + st_c * 16) = v;
        }
    }
}

// Two groups of wavefronts in a workgroup (GROUPS == 2): what the second has summed up
// goes through LDS - its own tiles, which nobody reads any more - to the first, which
// holds the same rows and adds it.  own: the group's array of the wavefront, 64 lanes x
// 16 * N values; BYTES from the first group's to the second's.
template<int N, int BYTES>
__device__ __forceinline__ void bwd_add_groups(int grp, char *own, f32x16 (&acc)[N])
{
    static_assert(64 * 16 * N * 4 == BYTES, "a wavefront's sums fill its array");
    float *at = reinterpret_cast<float *>(own + (grp == 0 ? BYTES : 0)) + lane_index_again();
    if(grp == 1)
    {
#pragma unroll
        for(int db = 0; db < N; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                at[(16 * db + r) * 64] = acc[db][r];
            }
        }
    }
    __syncthreads();
    if(grp == 0)
    {
#pragma unroll
        for(int db = 0; db < N; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                acc[db][r] += at[(16 * db + r) * 64];
            }
        }
    }
}

// Two wavefronts that halved the steps of the same 32 rows (KH == 2): each gives the
// other the blocks of its sums that lie in the other's half of the head - those behind
// N in acc - and adds what it gets to its own.  own, theirs: an array of LDS each.
template<int N>
__device__ __forceinline__ void bwd_add_halves(char *own, const char *theirs, f32x16 (&acc)[2 * N])
{
    const int lane = lane_index_again();
    float *to = reinterpret_cast<float *>(own) + lane;
    const float *from = reinterpret_cast<const float *>(theirs) + lane;
#pragma unroll
    for(int db = 0; db < N; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            to[(16 * db + r) * 64] = acc[N + db][r];
        }
    }
    __syncthreads();
#pragma unroll
    for(int db = 0; db < N; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            acc[db][r] += from[(16 * db + r) * 64];
        }
    }
}

// KH: 2: the workgroup has 64 rows, and each step's 64 are shared by two wavefronts of
// the same 32 rows, 32 each (see the launcher).
// GROUPS: 2: the workgroup is two groups of four wavefronts on the same rows, which
// take the steps of the walk in turn through tiles of their own (see the launcher).
// GRID: the rows of both sequence axes live in separately allocated tiles
// (BwdGridParams); a workgroup's own 128 rows lie in one tile and every 64-row
// step of the other axis does too, because tile sizes are multiples of 128.
template<typename T, int HEAD, int MODE, bool GRID, int GROUPS, int KH, bool OWN>
__device__ __forceinline__ void sdpa_bwd_dq_body(
        const std::conditional_t<GRID, BwdGridParams, BwdParams> &p, unsigned wg,
        char *lds_k0, char *lds_k1, char *lds_v0, char *lds_v1, uint32_t *lds_word)
{
    typedef typename T::vec8 vec8;
    typedef BwdTile<HEAD> G;
    constexpr int KSTEPS = G::KSTEPS, DBLOCKS = G::DBLOCKS, RB = G::RB, CPR = G::CPR;
    constexpr int LOADS_PER_WAVE = G::LOADS_PER_WAVE, ROWS_PER_LOAD = G::ROWS_PER_LOAD;
    constexpr bool EXPLICIT = (MODE == NNTILE_HIP_MASK_ADDITIVE
            || MODE == NNTILE_HIP_MASK_BOOL);

    const int tid = (int)threadIdx.x % kBwdThreads;
    const int grp = GROUPS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kBwdThreads) : 0;
    // (the group's half of every array in LDS: part of the lanes' read addresses)
    const int lds_grp = grp * G::BYTES;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    constexpr int ROWS = kBwdRows / KH;     // queries of the workgroup
    constexpr int NB = 2 / KH;              // 32-key blocks of a step that a wavefront takes
    const int rows32 = KH > 1 ? wave_u & 1 : wave_u;    // which of the workgroup's queries
    const int kh = KH > 1 ? wave_u >> 1 : 0;            // which 32 keys of a step
    const int col = lane & 31;
    const int half = lane >> 5;

    const int q_blocks = (int)((p.q_seq + ROWS - 1) / ROWS);
    // the last query blocks see the most keys under a causal mask: first
    int b, q_block;
    // (the grid form: the slab of the entry, whose tiles are allocations of
    // their own)
    int q_tile0 = 0, k_tile0 = 0;
    int64_t d_slab = 0;
    if constexpr(GRID)
    {
        map_workgroup(wg, p.batch * p.n_slabs, q_blocks, true, b, q_block);
        if(p.n_slabs > 1)
        {
            const int slab = b / p.batch;
            b -= slab * p.batch;
            q_tile0 = slab * p.n_q_tiles;
            k_tile0 = slab * p.n_kv_tiles;
            d_slab = (int64_t)slab * p.q_seq * p.batch;
        }
    }
    else
    {
        map_workgroup(wg, p.batch, q_blocks, true, b, q_block);
    }
    const int q_row0 = q_block * ROWS;
    const int kvb = kv_entry(b, p.n_batch, p.kv_group);
    const int q_seq = (int)p.q_seq, k_seq = (int)p.k_seq;
    const int my_q = q_row0 + rows32 * 32 + col;
    const bool q_ok = my_q < q_seq;
    // the lane's query: its row within the allocation that holds it (of Q, dA,
    // dQ, and of lse without the head axis), and its place among the row dots
    // (a function of the row, so that the stores at the end can work it out
    // again instead of keeping it through the loop)
    int own_t0 = 0, own_rows = q_seq;           // the tile that holds the block's rows
    if constexpr(GRID)
    {
        const int q_tile = (int)p.q_tile;
        own_t0 = __builtin_amdgcn_readfirstlane((q_row0 / q_tile) * q_tile);
        own_rows = min(q_tile, q_seq - own_t0);
    }
    auto row_elem = [&](int row, bool ok) __attribute__((always_inline)) -> int64_t
    {
        return (int64_t)b * own_rows + ((ok ? row : (GRID ? q_row0 : 0)) - own_t0);
    };
    const int64_t q_elem = row_elem(my_q, q_ok);
    int64_t d_idx = q_elem;
    const void *Q_own = p.Q, *dA_own = p.dA;
    void *dQ_own = p.dQ;
    const float *lse_own = p.lse;
    if constexpr(GRID)
    {
        const int q_tile = (int)p.q_tile;
        const int tq = q_row0 / q_tile, t0 = tq * q_tile;
        d_idx = d_slab + (int64_t)p.batch * t0 + q_elem;
        Q_own = p.Qt[q_tile0 + tq];
        dA_own = p.dAt[q_tile0 + tq];
        dQ_own = p.dQt[q_tile0 + tq];
        lse_own = p.lset[q_tile0 + tq];
    }
    const int64_t q_off = q_elem * HEAD;

    // Q and dA fragments (B operands); the row dot D = dA . A of the query
    vec8 qf[KSTEPS], gf[KSTEPS];
    {
        const uint16_t *qs = static_cast<const uint16_t *>(Q_own) + q_off + half * 8;
        const uint16_t *gs = static_cast<const uint16_t *>(dA_own) + q_off + half * 8;
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            u32x4 q = *reinterpret_cast<const u32x4 *>(qs + ks * 16);
            u32x4 g = *reinterpret_cast<const u32x4 *>(gs + ks * 16);
            if(!q_ok)
            {
                q = u32x4{0, 0, 0, 0};
                g = u32x4{0, 0, 0, 0};
            }
            qf[ks] = __builtin_bit_cast(vec8, q);
            gf[ks] = __builtin_bit_cast(vec8, g);
        }
    }
    float d_row;
    if constexpr(OWN)
    {
        // (a lane's fragments are every second eight of its row: the sums in the order
        // of the exchanges that add them up in the launch in front)
        const uint16_t *as = static_cast<const uint16_t *>(p.A) + q_off + half * 8;
        float part[KSTEPS];
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            part[ks] = bwd_dot8<T>(__builtin_bit_cast(u32x4, gf[ks]),
                    *reinterpret_cast<const u32x4 *>(as + ks * 16));
        }
#pragma unroll
        for(int o = KSTEPS / 2; o >= 1; o /= 2)
        {
#pragma unroll
            for(int ks = 0; ks < o; ++ks)
            {
                part[ks] += part[ks + o];
            }
        }
        d_row = part[0] + __shfl_xor(part[0], 32, 64);
        d_row = q_ok ? d_row : 0.0f;
    }
    else
    {
        d_row = q_ok ? p.D[d_idx] : 0.0f;
    }
    const float lse_q = q_ok ? lse_own[q_elem] : neg_inf();
    // exponent offset in log2 units; a row that saw nothing has P = 0
    const float lse2 = (lse_q == neg_inf()) ? __builtin_huge_valf() : lse_q * kLog2e;

    // ---- which keys ---------------------------------------------------------------
    // key row kg is visible to query row q iff kg <= rel + q (causal)
    // (a mask given as values: the rule its blocks are compared with)
    int64_t rel64 = EXPLICIT ? 0 : p.q_pos0 + p.causal_offset - p.k_pos0;
    rel64 = max((int64_t)-(1 << 30), min(rel64, (int64_t)(1 << 30)));
    const int rel = (int)rel64;
    int n_steps = (k_seq + kBwdStep - 1) / kBwdStep;
    if(MODE == NNTILE_HIP_MASK_CAUSAL)
    {
        const int hi = min(rel + min(q_row0 + ROWS, q_seq) - 1, k_seq - 1);
        n_steps = hi < 0 ? 0 : min(n_steps, hi / kBwdStep + 1);
    }
    const int my_lim = rel + my_q;          // last visible key of this lane's query

    // ---- LDS addresses --------------------------------------------------------------
    uint32_t ld_goff[LOADS_PER_WAVE];
    const int ld_cpos = lane % CPR;
    const int ld_row0 = wave * LOADS_PER_WAVE * ROWS_PER_LOAD + lane / CPR;   // + i * ROWS_PER_LOAD
#pragma unroll
    for(int i = 0; i < LOADS_PER_WAVE; ++i)
    {
        const int r = ld_row0 + i * ROWS_PER_LOAD;
        ld_goff[i] = (uint32_t)(r * RB + (ld_cpos ^ G::swz(r)) * 16);
    }
    // (only the last step of the keys can be short: its rows past the end read
    // the last row that exists; the offsets of that step are kept beside the
    // others rather than computed per load)
    uint32_t ld_goff_end[LOADS_PER_WAVE];
    {
        const int last_of_end = (k_seq - 1) % kBwdStep;
#pragma unroll
        for(int i = 0; i < LOADS_PER_WAVE; ++i)
        {
            ld_goff_end[i] = ld_goff[i]
                - (uint32_t)(max(ld_row0 + i * ROWS_PER_LOAD - last_of_end, 0) * RB);
        }
    }
    // row operand: lane (col, half) reads row mb*32+col, logical chunk 2*ks+half;
    // 32 rows further on the swizzle is the same, so mb goes into the immediate
    uint32_t row_raddr[KSTEPS];
#pragma unroll
    for(int ks = 0; ks < KSTEPS; ++ks)
    {
        row_raddr[ks] = (uint32_t)(lds_grp + (kh * 32 + col) * RB + ((2 * ks + half) ^ G::swz(col)) * 16);
    }
    // transposed operand: within a 16-lane block lane i addresses row j = i/4 and
    // head values 4*(i%4)..+3 of the block's 16; lanes 16..31 take the upper 16
    // head values of a 32-row block, the lane half the rows 4..7.  For the
    // 16-row sub-step t the two reads cover rows 16t + 4*half + j and + 8; the
    // swizzle of a row does not depend on t, so 16t goes into the immediate.
    uint32_t tr_raddr[2][DBLOCKS];
    {
        const int i16 = lane & 15, dblk = (lane >> 4) & 1;
        const int j = i16 >> 2, r4 = i16 & 3;
#pragma unroll
        for(int a = 0; a < 2; ++a)
        {
            const int r = 4 * half + j + 8 * a;
#pragma unroll
            for(int db = 0; db < DBLOCKS; ++db)
            {
                // (KH == 2: the blocks that the wavefront is left with come first)
                const int c = 4 * ((db + kh * (DBLOCKS / 2)) % DBLOCKS) + 2 * dblk + (r4 >> 1);
                tr_raddr[a][db] = (uint32_t)(lds_grp + (kh * 32 + r) * RB + (c ^ G::swz(r)) * 16 + 8 * (r4 & 1));
            }
        }
    }

    const char *Kb = static_cast<const char *>(p.K) + (int64_t)kvb * k_seq * RB;
    const char *Vb = static_cast<const char *>(p.V) + (int64_t)kvb * k_seq * RB;
    // loads of key step g; rows past the end are clamped to the last row
    // (their probabilities are exactly 0)
    // (a wave gets one such load accepted every ~64 cycles and stands still
    // until then: inside the loop the loads go between the MFMAs, one K and
    // one V load at a time)
    struct KeyRows
    {
        const char *K, *V;      // the step's first row of the entry
        bool at_end;
    };
    auto key_rows = [&](int g) __attribute__((always_inline)) -> KeyRows
    {
        const int row0 = g * kBwdStep;
        const bool at_end = row0 + kBwdStep > k_seq;
        if constexpr(GRID)
        {
            const int k_tile = (int)p.k_tile;
            const int tk = row0 / k_tile, t0 = tk * k_tile;
            const int64_t off = ((int64_t)kvb * min(k_tile, k_seq - t0) + (row0 - t0)) * RB;
            return KeyRows{static_cast<const char *>(p.Kt[k_tile0 + tk]) + off,
                static_cast<const char *>(p.Vt[k_tile0 + tk]) + off, at_end};
        }
        else
        {
            return KeyRows{Kb + (int64_t)row0 * RB, Vb + (int64_t)row0 * RB, at_end};
        }
    };
    auto fetch_piece = [&](const KeyRows &at, char *kdst_base, char *vdst_base, int i)
        __attribute__((always_inline))
    {
        char *kdst = kdst_base + lds_grp + wave_u * LOADS_PER_WAVE * 1024;
        char *vdst = vdst_base + lds_grp + wave_u * LOADS_PER_WAVE * 1024;
        const uint32_t goff = at.at_end ? ld_goff_end[i] : ld_goff[i];
        load_to_lds16<0, false>(at.K, goff, kdst + i * 1024);
        load_to_lds16<0, false>(at.V, goff, vdst + i * 1024);
    };
    auto fetch = [&](int g, char *kdst_base, char *vdst_base)
    {
        const KeyRows at = key_rows(g);
#pragma unroll
        for(int i = 0; i < LOADS_PER_WAVE; ++i)
        {
            fetch_piece(at, kdst_base, vdst_base, i);
        }
    };
    constexpr int FETCH_STRIDE = (NNTILE_BWD_SPREAD == 2 ? NB : 1) * KSTEPS / LOADS_PER_WAVE;
    static_assert(FETCH_STRIDE >= 1 && 1 + (LOADS_PER_WAVE - 1) * FETCH_STRIDE < NB * KSTEPS,
            "the pieces of a fetch must fit between the MFMAs of a step");

    f32x16 acc[DBLOCKS];
#pragma unroll
    for(int db = 0; db < DBLOCKS; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            acc[db][r] = 0.0f;
        }
    }
    const float c = p.scale * kLog2e;
    // mask values: the workgroup's first row of the mask, and the byte offset
    // of the lane's row from there (the launcher keeps 128 rows of the mask
    // within 32 bits); mask_off is that of the lane's first key in a step
    constexpr uint32_t MASK_ES = MODE == NNTILE_HIP_MASK_ADDITIVE ? 2u : 1u;
    const char *mask_wg = static_cast<const char *>(p.mask)
        + (int64_t)q_row0 * p.mask_ld * (int64_t)MASK_ES;
    const uint32_t mask_row_off = (uint32_t)(q_ok ? my_q - q_row0 : 0) * (uint32_t)p.mask_ld * MASK_ES;
    // (at head 128 the groups of four cost registers that the body does not have)
    constexpr bool MASK_GROUPS = HEAD <= 64;
    const uint32_t mask_off_wg = mask_row_off + (uint32_t)(kh * 32 + 4 * half) * MASK_ES;

    // the workgroup's two query blocks of 64 against the key blocks 0 .. n_steps-1
    constexpr bool OWN_CLASSES = OWN && EXPLICIT;
    const uint32_t own_bits = OWN_CLASSES ? bwd_own_classes<T, MODE>(p, q_row0 / kBwdStep, 0, n_steps, true,
            lds_word) : 0u;
    const StepSet steps = make_step_set(p, EXPLICIT, q_row0 / kBwdStep,
            min(ROWS / kBwdStep, (q_seq - q_row0 + kBwdStep - 1) / kBwdStep), 0, n_steps, true,
            OWN_CLASSES, own_bits);
    // (the group's steps: every second of the walk)
    auto next_own = [&](int g) __attribute__((always_inline)) -> int
    {
        const int n = steps.next(g);
        return GROUPS == 1 || n < 0 ? n : steps.next(n);
    };
    int g_cur = steps.begin(), g_last = -1;
    if(GROUPS > 1 && grp == 1 && g_cur >= 0)
    {
        g_last = -2;                        // (the first group has a step)
        g_cur = steps.next(g_cur);
    }
    if(g_cur >= 0)
    {
        fetch(g_cur, lds_k0, lds_v0);
    }
    // masked_tag: the step reads mask values (as a compile-time choice, so
    // that the reads of a step stay one batch of loads)
    auto step = [&](int g, int g_next, auto buf_tag, auto masked_tag)
        __attribute__((always_inline))
    {
        constexpr int BUF = decltype(buf_tag)::value;
        const char *Ks = BUF ? lds_k1 : lds_k0;
        const char *Vs = BUF ? lds_v1 : lds_v0;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // the last step loads its own tile once more, rather than branch
        // (wave-common, computed once here: the loads between the MFMAs below
        // only add their offsets)
        const KeyRows at_f = key_rows(g_next >= 0 ? g_next : g);
        if(NNTILE_BWD_SPREAD == 0 && g_next >= 0)
        {
            fetch(g_next, BUF ? lds_k0 : lds_k1, BUF ? lds_v0 : lds_v1);
        }
        constexpr bool use_mask = EXPLICIT && decltype(masked_tag)::value;
        const int kg0 = g * kBwdStep;
        const int keys_here = min(kBwdStep, k_seq - kg0);
        // (groups of four: offsets count from four keys in front of the step -
        // where there are keys in front - as a step of fewer than four keys is
        // read from there on)
        const uint32_t lead = MASK_GROUPS && kg0 > 0 ? 4u * MASK_ES : 0u;
        const char *mask_step = mask_wg + (int64_t)kg0 * MASK_ES - lead;
        // (the last place that a group of values, or a value, can start at)
        const uint32_t mask_off_last = mask_row_off + lead
            + (uint32_t)(keys_here - (MASK_GROUPS ? 4 : 1)) * MASK_ES;
        // (through an empty asm statement: the 32 offsets that a step adds
        // constants to are then made where the step uses them instead of once
        // before the loop and kept, which at head 128 means spilled)
        uint32_t mask_off = mask_off_wg + lead;
        if(use_mask)
        {
            asm volatile("" : "+v"(mask_off));
        }

        // ---- S^T = K Q^T, dP^T = V dA^T -------------------------------------------------
        // (one 32-key block at a time: half the accumulators live)
        // ---- P^T, dS^T: register r of block mb is key mb*32 + tile_row(r, half) ------------
        int lim = keys_here - 1;
        // (the mask of this step is the rule `key <= query + rel`)
        const bool ruled = MODE == NNTILE_HIP_MASK_CAUSAL
            || (EXPLICIT && !use_mask && !steps.is_open(g));
        if(ruled)
        {
            lim = min(lim, my_lim - kg0);
        }
        const int lim_less_half = lim - 4 * half - kh * 32;
        // (wave-common: the last key of the step against the last key that
        // exists and the last key the workgroup's first query sees)
        const bool bounds = keys_here < kBwdStep
            || (ruled && kg0 + kBwdStep - 1 > rel + q_row0);
        if constexpr(use_mask || NNTILE_BWD_PIPE_DQ == 0)
        {
#pragma unroll
            for(int mb = 0; mb < NB; ++mb)
            {
                f32x16 sv, dpv;
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    sv[r] = 0.0f;
                    dpv[r] = 0.0f;
                }
#pragma unroll
                for(int ks = 0; ks < KSTEPS; ++ks)
                {
                    const vec8 ka = *reinterpret_cast<const vec8 *>(Ks + row_raddr[ks] + mb * 32 * RB);
                    const vec8 va = *reinterpret_cast<const vec8 *>(Vs + row_raddr[ks] + mb * 32 * RB);
                    sv = T::mfma(ka, qf[ks], sv);
                    dpv = T::mfma(va, gf[ks], dpv);
#pragma unroll
                    for(int j = 0; j < LOADS_PER_WAVE; ++j)
                    {
                        if(NNTILE_BWD_SPREAD != 0 && mb * KSTEPS + ks == 1 + j * FETCH_STRIDE)
                        {
                            fetch_piece(at_f, BUF ? lds_k0 : lds_k1, BUF ? lds_v0 : lds_v1, j);
                        }
                    }
                }
                // Keys past the end and keys the causal mask hides: their scores
                // become -inf in a pass of their own, which only the steps at the
                // end of the keys and on the diagonal run (a wave-common branch).
                if(bounds)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        // (key mb*32 + tile_row(r, half) <= lim, the lane's part on the right)
                        sv[r] = mb * 32 + tile_row(r, 0) <= lim_less_half ? sv[r] : neg_inf();
                    }
                }
                // The values of four consecutive keys in one load of any
                // alignment (2-byte loads, each touching 32 rows, took most of
                // a masked step): wave-common address of the step's first key in
                // the workgroup's first row + the lane's 32-bit offset.  A group
                // that would reach past the row is moved back to end with it and
                // shifted into place; keys past the end are hidden above.
                uint64_t mval[4] = {0, 0, 0, 0};
                if constexpr(use_mask && MASK_GROUPS)
                {
                    typedef std::conditional_t<MODE == NNTILE_HIP_MASK_ADDITIVE, uint64_t,
                            uint32_t> group_t;
                    typedef group_t __attribute__((aligned(1))) group_any;
#pragma unroll
                    for(int rg = 0; rg < 4; ++rg)
                    {
                        const uint32_t want = mask_off + (uint32_t)(mb * 32 + 8 * rg) * MASK_ES;
                        const uint32_t at = min(want, mask_off_last);
                        if(k_seq >= 4)
                        {
                            mval[rg] = (uint64_t)*reinterpret_cast<const group_any *>(
                                    mask_step + at) >> (8u * min(want - at, 7u));
                        }
                        else
                        {
                            // (rows of less than one group: the lane's first)
#pragma unroll
                            for(int e = 0; mb == 0 && rg == 0 && e < 3; ++e)
                            {
                                const char *mp = mask_step + mask_row_off
                                    + (uint32_t)min(e, k_seq - 1) * MASK_ES;
                                const uint32_t x = (MODE == NNTILE_HIP_MASK_ADDITIVE)
                                    ? *reinterpret_cast<const uint16_t *>(mp)
                                    : *reinterpret_cast<const uint8_t *>(mp);
                                mval[rg] |= (uint64_t)x << (8 * MASK_ES * e);
                            }
                        }
                    }
                }
                float dsv[16];
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    float e = fmaf(sv[r], c, -lse2);        // -inf: hidden, or a row that saw nothing
                    bool visible = true;
                    if(use_mask)
                    {
                        uint32_t x;
                        if constexpr(MASK_GROUPS)
                        {
                            x = (uint32_t)(mval[r / 4] >> (8 * MASK_ES * (r % 4)))
                                & (MODE == NNTILE_HIP_MASK_ADDITIVE ? 0xffffu : 0xffu);
                        }
                        else
                        {
                            const char *mp = mask_step + min(mask_off
                                    + (uint32_t)(mb * 32 + tile_row(r, 0)) * MASK_ES, mask_off_last);
                            x = (MODE == NNTILE_HIP_MASK_ADDITIVE)
                                ? *reinterpret_cast<const uint16_t *>(mp)
                                : *reinterpret_cast<const uint8_t *>(mp);
                        }
                        if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                        {
                            const float add = T::to_float((uint16_t)x);
                            visible = visible && (add != neg_inf());
                            e = fmaf(add, kLog2e, e);
                        }
                        else
                        {
                            visible = visible && (x != 0);
                        }
                    }
                    const float pr = use_mask ? (visible ? fast_exp2(e) : 0.0f) : fast_exp2(e);
                    dsv[r] = pr * (dpv[r] - d_row);
                }
                uint32_t ds_pk[8];
#pragma unroll
                for(int k = 0; k < 8; ++k)
                {
                    ds_pk[k] = T::pack2(dsv[2 * k], dsv[2 * k + 1]);
                }
                // ---- dQ^T += K^T dS^T: the block's two sub-steps of 16 keys ------------------
#pragma unroll
                for(int tt = 0; tt < 2; ++tt)
                {
                    const int t = 2 * mb + tt;
                    const u32x4 braw = {ds_pk[4 * tt], ds_pk[4 * tt + 1], ds_pk[4 * tt + 2],
                        ds_pk[4 * tt + 3]};
                    const vec8 bop = __builtin_bit_cast(vec8, braw);
#pragma unroll
                    for(int db = 0; db < DBLOCKS; ++db)
                    {
                        const u32x2 lo = bwd_lds_read_tr16(Ks + tr_raddr[0][db] + (16 * t) * RB);
                        const u32x2 hi = bwd_lds_read_tr16(Ks + tr_raddr[1][db] + (16 * t) * RB);
                        const u32x4 araw = {lo[0], lo[1], hi[0], hi[1]};
                        acc[db] = T::mfma(__builtin_bit_cast(vec8, araw), bop, acc[db]);
                    }
                }
            }
        }
        else if constexpr(KH > 1)
        {
            // One block of 32 keys: S^T, dP^T with the exponentials beside it, dS^T, then
            // dQ^T += K^T dS^T, in slots as below.
            f32x16 sv, dpv;
            uint32_t ds_pk[8];
            constexpr int SLOTS = 2 * KSTEPS + 2 * DBLOCKS;
            constexpr int AHEAD = kBwdAhead<HEAD>;
            vec8 ring[AHEAD + 1];
            auto read = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g < 2 * KSTEPS)
                {
                    ring[g % (AHEAD + 1)] = *reinterpret_cast<const vec8 *>((g < KSTEPS ? Ks : Vs)
                            + row_raddr[g % KSTEPS]);
                }
                else if constexpr(g < SLOTS)
                {
                    constexpr int i = g - 2 * KSTEPS, t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x2 lo = bwd_lds_read_tr16(Ks + tr_raddr[0][db] + (16 * t) * RB);
                    const u32x2 hi = bwd_lds_read_tr16(Ks + tr_raddr[1][db] + (16 * t) * RB);
                    const u32x4 araw = {lo[0], lo[1], hi[0], hi[1]};
                    ring[g % (AHEAD + 1)] = __builtin_bit_cast(vec8, araw);
                }
            };
            each_slot(read, std::make_integer_sequence<int, AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            each_slot([&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g == KSTEPS)
                {
                    // (keys past the end and keys the rule hides: see below)
                    if(bounds)
                    {
#pragma unroll
                        for(int r = 0; r < 16; ++r)
                        {
                            sv[r] = tile_row(r, 0) <= lim_less_half ? sv[r] : neg_inf();
                        }
                    }
                }
                if constexpr(g == 2 * KSTEPS)
                {
#pragma unroll
                    for(int k = 0; k < 8; ++k)
                    {
                        ds_pk[k] = T::pack2(sv[2 * k] * (dpv[2 * k] - d_row),
                                sv[2 * k + 1] * (dpv[2 * k + 1] - d_row));
                    }
                }
                read(std::integral_constant<int, g + AHEAD>{});
                const vec8 a = ring[g % (AHEAD + 1)];
                if constexpr(g < KSTEPS)
                {
                    sv = T::mfma(a, qf[g], g == 0 ? f32x16{} : sv);
#pragma unroll
                    for(int j = 0; j < LOADS_PER_WAVE; ++j)
                    {
                        if(NNTILE_BWD_SPREAD != 0 && g == 1 + j * FETCH_STRIDE)
                        {
                            fetch_piece(at_f, BUF ? lds_k0 : lds_k1, BUF ? lds_v0 : lds_v1, j);
                        }
                    }
                }
                else if constexpr(g < 2 * KSTEPS)
                {
                    constexpr int i = g - KSTEPS;
                    dpv = T::mfma(a, gf[i], i == 0 ? f32x16{} : dpv);
#pragma unroll
                    for(int r = i * 16 / KSTEPS; r < (i + 1) * 16 / KSTEPS; ++r)
                    {
                        // (-inf: hidden, or a row that saw nothing)
                        sv[r] = fast_exp2(fmaf(sv[r], c, -lse2));
                    }
                }
                else
                {
                    constexpr int i = g - 2 * KSTEPS, t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x4 braw = {ds_pk[4 * t], ds_pk[4 * t + 1], ds_pk[4 * t + 2],
                        ds_pk[4 * t + 3]};
                    acc[db] = T::mfma(a, __builtin_bit_cast(vec8, braw), acc[db]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, SLOTS>{});
        }
        else
        {
            // The step's two 32-key blocks in three phases each - A: the two
            // score products, B: dS on the vector ALU, C: dQ^T += K^T dS^T -
            // issued as A0 | A1 with B0 | C0 with B1 | C1 (see the dK / dV body):
            // slots of one MFMA, the operand read of the slot AHEAD later (across
            // the phases' borders too) and a slice of the vector work, with a
            // scheduling barrier after each.
            f32x16 sv[2], dpv[2];
            uint32_t ds_pk[2][8];
            constexpr int A_MFMAS = 2 * KSTEPS, C_MFMAS = 2 * DBLOCKS;
            constexpr int SLOTS = 2 * (A_MFMAS + C_MFMAS);
            constexpr int AHEAD = kBwdAhead<HEAD>;
            vec8 ring[AHEAD + 1];
            auto read = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g < 2 * A_MFMAS)
                {
                    constexpr int mb = g / A_MFMAS, i = g % A_MFMAS;
                    ring[g % (AHEAD + 1)] = *reinterpret_cast<const vec8 *>(((i & 1) ? Vs : Ks)
                            + row_raddr[i / 2] + mb * 32 * RB);
                }
                else if constexpr(g < SLOTS)
                {
                    constexpr int i = g - 2 * A_MFMAS, t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x2 lo = bwd_lds_read_tr16(Ks + tr_raddr[0][db] + (16 * t) * RB);
                    const u32x2 hi = bwd_lds_read_tr16(Ks + tr_raddr[1][db] + (16 * t) * RB);
                    const u32x4 araw = {lo[0], lo[1], hi[0], hi[1]};
                    ring[g % (AHEAD + 1)] = __builtin_bit_cast(vec8, araw);
                }
            };
            auto mfma = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                const vec8 a = ring[g % (AHEAD + 1)];
                if constexpr(g < 2 * A_MFMAS)
                {
                    constexpr int mb = g / A_MFMAS, i = g % A_MFMAS, ks = i / 2;
                    if constexpr((i & 1) == 0)
                    {
                        sv[mb] = T::mfma(a, qf[ks], ks == 0 ? f32x16{} : sv[mb]);
                    }
                    else
                    {
                        dpv[mb] = T::mfma(a, gf[ks], ks == 0 ? f32x16{} : dpv[mb]);
#pragma unroll
                        for(int j = 0; j < LOADS_PER_WAVE; ++j)
                        {
                            if(NNTILE_BWD_SPREAD != 0 && mb * KSTEPS + ks == 1 + j * FETCH_STRIDE)
                            {
                                fetch_piece(at_f, BUF ? lds_k0 : lds_k1, BUF ? lds_v0 : lds_v1, j);
                            }
                        }
                    }
                }
                else
                {
                    constexpr int i = g - 2 * A_MFMAS, mb = i / C_MFMAS;
                    constexpr int tt = i % C_MFMAS / DBLOCKS, db = i % DBLOCKS;
                    const u32x4 braw = {ds_pk[mb][4 * tt], ds_pk[mb][4 * tt + 1],
                        ds_pk[mb][4 * tt + 2], ds_pk[mb][4 * tt + 3]};
                    acc[db] = T::mfma(a, __builtin_bit_cast(vec8, braw), acc[db]);
                }
            };
            // Keys past the end and keys the causal mask hides: their scores
            // become -inf in a pass of their own, which only the steps at the
            // end of the keys and on the diagonal run (a wave-common branch).
            auto hide = [&](int mb) __attribute__((always_inline))
            {
                if(bounds)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        // (key mb*32 + tile_row(r, half) <= lim, the lane's part on the right)
                        sv[mb][r] = mb * 32 + tile_row(r, 0) <= lim_less_half ? sv[mb][r]
                            : neg_inf();
                    }
                }
            };
            float ds_even = 0.0f;
            auto b_item = [&](int mb, int r) __attribute__((always_inline))
            {
                const float e = fmaf(sv[mb][r], c, -lse2);        // -inf: hidden, or a row that saw nothing
                const float pr = fast_exp2(e);
                const float dsr = pr * (dpv[mb][r] - d_row);
                if(r % 2 == 0)
                {
                    ds_even = dsr;
                }
                else
                {
                    ds_pk[mb][r / 2] = T::pack2(ds_even, dsr);
                    asm volatile("" : "+v"(ds_pk[mb][r / 2]));
                }
            };
            each_slot(read, std::make_integer_sequence<int, AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            each_slot([&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                constexpr int i1 = g - A_MFMAS, i2 = g - 2 * A_MFMAS;
                if constexpr(i1 == 0)
                {
                    hide(0);
                }
                if constexpr(i2 == 0)
                {
                    hide(1);
                }
                read(std::integral_constant<int, g + AHEAD>{});
                mfma(slot);
                if constexpr(i1 >= 0 && i1 < A_MFMAS)
                {
#pragma unroll
                    for(int r = i1 * 16 / A_MFMAS; r < (i1 + 1) * 16 / A_MFMAS; ++r)
                    {
                        b_item(0, r);
                    }
                }
                if constexpr(i2 >= 0 && i2 < C_MFMAS)
                {
#pragma unroll
                    for(int r = i2 * 16 / C_MFMAS; r < (i2 + 1) * 16 / C_MFMAS; ++r)
                    {
                        b_item(1, r);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, SLOTS>{});
        }
    };
    auto run = [&](int g, int g_next, auto buf_tag) __attribute__((always_inline))
    {
        if(EXPLICIT && !steps.is_open(g) && !steps.is_rule(g))
        {
            step(g, g_next, buf_tag, std::true_type{});
        }
        else
        {
            step(g, g_next, buf_tag, std::false_type{});
        }
    };
    while(g_cur >= 0)
    {
        int g_next = next_own(g_cur);
        run(g_cur, g_next, std::integral_constant<int, 0>{});
        g_last = g_cur;
        g_cur = g_next;
        if(g_cur < 0)
        {
            break;
        }
        g_next = next_own(g_cur);
        run(g_cur, g_next, std::integral_constant<int, 1>{});
        g_last = g_cur;
        g_cur = g_next;
    }
    // (the last step's spare loads into LDS must have landed before the
    // workgroup's LDS can be given away)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // (one barrier a step: the second group meets that of a last step it has not)
    if(GROUPS > 1 && grp == 1 && (g_last == -2 || (g_last >= 0 && steps.next(g_last) >= 0)))
    {
        __syncthreads();
    }

    // ---- dQ (+)= scale acc (every wavefront is done with the tiles in LDS) -----------
    __syncthreads();
    const int row_first = q_row0 + rows32 * 32;
    char *xch = (wave_u == 0 ? lds_k0 : wave_u == 1 ? lds_k1 : wave_u == 2 ? lds_v0 : lds_v1) + lds_grp;
    if constexpr(GROUPS > 1)
    {
        bwd_add_groups<DBLOCKS, G::BYTES>(grp, xch, acc);
        if(grp == 1)
        {
            return;
        }
    }
    if constexpr(KH > 1)
    {
        const char *other = wave_u == 0 ? lds_v0 : wave_u == 1 ? lds_v1 : wave_u == 2 ? lds_k0 : lds_k1;
        bwd_add_halves<DBLOCKS / 2>(xch, other, acc);
        xch += G::BYTES - 32 * (RB / 2);        // (behind what the other may still be reading)
    }
    bwd_store_rows<T, HEAD, KH>(xch, static_cast<char *>(dQ_own) + row_elem(row_first, true) * RB
            + kh * (RB / 2), q_seq - row_first, acc, p.scale, !p.overwrite);
}

// ---------------------------------------------------------------------------------
// PART says which gradient: K and V fragments plus both accumulators take 192
// registers of a lane at head 128, which leaves too few for two wavefronts
// per SIMD to run without spilling and without room to read operands ahead.
// One set of workgroups per gradient (dK: S, dP, dK^T; dV: S, dV^T - the
// scores are computed once more) fits two workgroups of 4 wavefronts on a CU.
enum { BWD_PART_DK = 1, BWD_PART_DV = 2 };
// Where one workgroup holds both gradients of its keys: at head sizes up to 64
// under every mask mode; at head 128 (K and V fragments and the two
// accumulators are 192 of a lane's 256 registers there) under the analytic
// modes, with the blocks of a step one after the other, product by product.
#ifndef NNTILE_BWD_FUSED_KEYS_HEAD
#define NNTILE_BWD_FUSED_KEYS_HEAD 64
#endif
#ifndef NNTILE_BWD_FUSED_KEYS_HEAD_ANALYTIC
#define NNTILE_BWD_FUSED_KEYS_HEAD_ANALYTIC 128
#endif
template<int HEAD, int MODE> constexpr bool kBwdFusedKeys = HEAD <= NNTILE_BWD_FUSED_KEYS_HEAD
    || (HEAD <= NNTILE_BWD_FUSED_KEYS_HEAD_ANALYTIC
            && (MODE == NNTILE_HIP_MASK_NONE || MODE == NNTILE_HIP_MASK_CAUSAL));
constexpr int kBwdCUs = 256;
constexpr int kDkvWaves = 4;
constexpr int kDkvThreads = kDkvWaves * 64;
constexpr int kDkvRows = kDkvWaves * 32;        // keys per workgroup

template<typename T, int HEAD, int MODE, int PART, bool GRID, int GROUPS, int KH, bool OWN>
__device__ __forceinline__ void sdpa_bwd_dkv_body(
        const std::conditional_t<GRID, BwdGridParams, BwdParams> &p, unsigned wg,
        char *lds_q0, char *lds_q1, char *lds_g0, char *lds_g1,
        float (*lds_stat)[2][kBwdStep], uint32_t *lds_word, float *lds_own)
{
    constexpr bool DO_DK = (PART & BWD_PART_DK) != 0, DO_DV = (PART & BWD_PART_DV) != 0;
    constexpr bool BOTH = DO_DK && DO_DV;
    BWD_TRACE_DECL
    typedef typename T::vec8 vec8;
    typedef BwdTile<HEAD> G;
    constexpr int KSTEPS = G::KSTEPS, DBLOCKS = G::DBLOCKS, RB = G::RB, CPR = G::CPR;
    constexpr int ROWS_PER_LOAD = G::ROWS_PER_LOAD;
    constexpr int LPW = G::LOADS >= kDkvWaves ? G::LOADS / kDkvWaves : 1;   // loads per loading wavefront
    constexpr int LOADERS = G::LOADS / LPW;                                  // wavefronts that load
    constexpr bool EXPLICIT = (MODE == NNTILE_HIP_MASK_ADDITIVE
            || MODE == NNTILE_HIP_MASK_BOOL);

    const int tid = (int)threadIdx.x % kDkvThreads;
    const int grp = GROUPS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kDkvThreads) : 0;
    // (the group's half of every array in LDS: part of the lanes' read addresses)
    const int lds_grp = grp * G::BYTES;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    constexpr int ROWS = kDkvRows / KH;     // keys of the workgroup
    constexpr int NB = 2 / KH;              // 32-query blocks of a step that a wavefront takes
    const int rows32 = KH > 1 ? wave_u & 1 : wave_u;    // which of the workgroup's keys
    const int kh = KH > 1 ? wave_u >> 1 : 0;            // which 32 queries of a step
    const int col = lane & 31;
    const int half = lane >> 5;

    const int q_seq = (int)p.q_seq, k_seq = (int)p.k_seq;
    const int k_blocks = (k_seq + ROWS - 1) / ROWS;
    // the first key blocks are seen by the most queries under a causal mask
    int kvb, k_block;                               // kvb = nb + n_batch*hkv
    int q_tile0 = 0, k_tile0 = 0;
    int64_t d_slab = 0;
    if constexpr(GRID)
    {
        const int kv_entries = p.batch / p.kv_group;
        map_workgroup(wg, kv_entries * p.n_slabs, k_blocks, false, kvb, k_block);
        if(p.n_slabs > 1)
        {
            const int slab = kvb / kv_entries;
            kvb -= slab * kv_entries;
            q_tile0 = slab * p.n_q_tiles;
            k_tile0 = slab * p.n_kv_tiles;
            d_slab = (int64_t)slab * p.q_seq * p.batch;
        }
    }
    else
    {
        map_workgroup(wg, p.batch / p.kv_group, k_blocks, false, kvb, k_block);
    }
    const int k_row0 = k_block * ROWS;
    const int nb = kvb % p.n_batch, hkv = kvb / p.n_batch;
    const int my_k = k_row0 + rows32 * 32 + col;
    const bool k_ok = my_k < k_seq;
    // key kg is visible to query q0 + qr + 4*half iff kg - 4*half <= rel + q0 + qr
    // (KH == 2: and q0 + 32 * kh)
    const int my_k_less_half = my_k - 4 * half - kh * 32;
    // the lane's key: its row within the allocation that holds it (of K, V, dK, dV)
    // (a function of the row, so that the stores at the end can work it out
    // again instead of keeping it through the loop)
    int own_t0 = 0, own_rows = k_seq;           // the tile that holds the block's rows
    if constexpr(GRID)
    {
        const int k_tile = (int)p.k_tile;
        own_t0 = __builtin_amdgcn_readfirstlane((k_row0 / k_tile) * k_tile);
        own_rows = min(k_tile, k_seq - own_t0);
    }
    auto row_elem = [&](int row, bool ok) __attribute__((always_inline)) -> int64_t
    {
        return (int64_t)kvb * own_rows + ((ok ? row : (GRID ? k_row0 : 0)) - own_t0);
    };
    const int64_t k_elem = row_elem(my_k, k_ok);
    const void *K_own = p.K, *V_own = p.V;
    void *dK_own = p.dK, *dV_own = p.dV;
    if constexpr(GRID)
    {
        const int k_tile = (int)p.k_tile;
        const int tk = k_row0 / k_tile;
        K_own = p.Kt[k_tile0 + tk];
        V_own = p.Vt[k_tile0 + tk];
        dK_own = p.dKt[k_tile0 + tk];
        dV_own = p.dVt[k_tile0 + tk];
    }
    const int64_t k_off = k_elem * HEAD;

    // K and V fragments (B operands): lane (col, half) holds head values 16*ks + 8*half..+7
    vec8 kf[KSTEPS], vf[KSTEPS];
    {
        const uint16_t *ks_ = static_cast<const uint16_t *>(K_own) + k_off + half * 8;
        const uint16_t *vs_ = static_cast<const uint16_t *>(V_own) + k_off + half * 8;
#pragma unroll
        for(int ks = 0; ks < KSTEPS; ++ks)
        {
            u32x4 k = *reinterpret_cast<const u32x4 *>(ks_ + ks * 16);
            u32x4 v = *reinterpret_cast<const u32x4 *>(vs_ + ks * 16);
            if(!k_ok)
            {
                k = u32x4{0, 0, 0, 0};
                v = u32x4{0, 0, 0, 0};
            }
            kf[ks] = __builtin_bit_cast(vec8, k);
            vf[ks] = __builtin_bit_cast(vec8, DO_DK ? v : u32x4{0, 0, 0, 0});
        }
    }

    // key row kg is visible to query row q iff kg <= rel + q (causal)
    // (a mask given as values: the rule its blocks are compared with)
    int64_t rel64 = EXPLICIT ? 0 : p.q_pos0 + p.causal_offset - p.k_pos0;
    rel64 = max((int64_t)-(1 << 30), min(rel64, (int64_t)(1 << 30)));
    const int rel = (int)rel64;
    const int n_steps = (q_seq + kBwdStep - 1) / kBwdStep;
    int first_step = 0;
    if(MODE == NNTILE_HIP_MASK_CAUSAL)
    {
        // the first query that sees the workgroup's first key
        const int q_lo = max(k_row0 - rel, 0);
        first_step = min(q_lo / kBwdStep, n_steps);
    }

    // (only the last step of the queries can be short: its rows past the end
    // read the last row that exists; the offsets of that step are kept beside
    // the others rather than computed per load)
    uint32_t ld_goff[LPW], ld_goff_end[LPW];
    const int ld_cpos = lane % CPR;
#pragma unroll
    for(int i = 0; i < LPW; ++i)
    {
        const int r = ((wave % LOADERS) * LPW + i) * ROWS_PER_LOAD + lane / CPR;
        ld_goff[i] = (uint32_t)(r * RB + (ld_cpos ^ G::swz(r)) * 16);
        ld_goff_end[i] = ld_goff[i] - (uint32_t)(max(r - (q_seq - 1) % kBwdStep, 0) * RB);
    }
    // Both gradients at head 128 leave no registers for the tables of offsets
    // here and below: one register stands for each table, an exclusive or with a
    // constant makes the entry where it is used (the chunk index of a row's
    // swizzled place is an exclusive or of the row's and the chunk's own bits).
    constexpr bool WIDE = BOTH && HEAD > 64 && KH == 1;
    static_assert(!WIDE || (CPR == 16 && ROWS_PER_LOAD == 4 && LPW == 4 && LOADERS == kDkvWaves
                && KSTEPS == 8 && DBLOCKS == 4), "the wide body's offsets are those of head 128");
    // (a load's rows 4j + lane / 16 of the wavefront's 16 have the swizzle of
    // lane / 16 with bits j)
    const uint32_t wide_goff = ld_goff[0];
    // row operand: lane (col, half) reads row mb*32+col, logical chunk 2*ks+half;
    // 32 rows further on the swizzle is the same, so mb goes into the immediate
    uint32_t row_raddr[KSTEPS];
#pragma unroll
    for(int ks = 0; ks < KSTEPS; ++ks)
    {
        row_raddr[ks] = (uint32_t)(lds_grp + (kh * 32 + col) * RB + ((2 * ks + half) ^ G::swz(col)) * 16);
    }
    uint32_t tr_raddr[2][DBLOCKS];
    {
        const int i16 = lane & 15, dblk = (lane >> 4) & 1;
        const int j = i16 >> 2, r4 = i16 & 3;
#pragma unroll
        for(int a = 0; a < 2; ++a)
        {
            const int r = 4 * half + j + 8 * a;
#pragma unroll
            for(int db = 0; db < DBLOCKS; ++db)
            {
                const int c = 4 * ((db + kh * (DBLOCKS / 2)) % DBLOCKS) + 2 * dblk + (r4 >> 1);
                tr_raddr[a][db] = (uint32_t)(lds_grp + (kh * 32 + r) * RB + (c ^ G::swz(r)) * 16 + 8 * (r4 & 1));
            }
        }
    }

    f32x16 dk[DBLOCKS], dv[DBLOCKS];
#pragma unroll
    for(int db = 0; db < DBLOCKS; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            dk[db][r] = 0.0f;
            dv[db][r] = 0.0f;
        }
    }
    const float c = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
                __builtin_bit_cast(int, p.scale * kLog2e)));
    // mask values: byte offsets of the lane's key within a row of the mask,
    // for the rows of the lower and of the upper half of the wave (the
    // launcher keeps 64 rows of the mask within 32 bits)
    constexpr uint32_t MASK_ES = MODE == NNTILE_HIP_MASK_ADDITIVE ? 2u : 1u;
    const uint32_t mask_row_bytes_wg = (uint32_t)p.mask_ld * MASK_ES;
    const uint32_t mask_off_lo = (uint32_t)(k_ok ? my_k : 0) * MASK_ES;
    const uint32_t mask_off_hi = mask_off_lo + (uint32_t)(4 * half) * mask_row_bytes_wg;
    // the workgroup's key blocks of 64 against the query blocks
    // first_step .. n_steps-1, once per head of the group: walk position
    // i = head * 64K + query step
    constexpr bool OWN_CLASSES = OWN && EXPLICIT;
    const uint32_t own_bits = OWN_CLASSES ? bwd_own_classes<T, MODE>(p, k_row0 / kBwdStep, first_step,
            n_steps, false, lds_word) : 0u;
    const StepSet steps = make_step_set(p, EXPLICIT, k_row0 / kBwdStep,
            min(ROWS / kBwdStep, (k_seq - k_row0 + kBwdStep - 1) / kBwdStep),
            first_step, n_steps, false, OWN_CLASSES, own_bits);
    constexpr int kHeadStride = 1 << 16;
    auto locate = [&](int i, int &bq, int &qs)
    {
        const int g = i / kHeadStride;
        qs = i % kHeadStride;
        bq = nb + p.n_batch * (g + p.kv_group * hkv);
    };
    auto walk_begin = [&]() -> int
    {
        return steps.begin();       // head 0
    };
    auto walk_next = [&](int i) -> int
    {
        const int g = i / kHeadStride;
        const int nxt = steps.next(i % kHeadStride);
        if(nxt >= 0)
        {
            return g * kHeadStride + nxt;
        }
        const int b0 = steps.begin();
        return (g + 1 < p.kv_group && b0 >= 0) ? (g + 1) * kHeadStride + b0 : -1;
    };
    // loads of walk position i: the Q and dA rows straight into LDS, the
    // logsumexp and D of its queries through registers (threads 0..127)
    // (inside the loop the tile loads go between the MFMAs, one Q and one dA
    // load at a time: a wave stands still ~64 cycles per load)
    // the allocation that holds query row0 of entry bq, the row's index in it
    // (for lse; times HEAD for Q and dA) and in the row dots
    struct QueryRows
    {
        const void *Q, *dA;
        const float *lse;
        int64_t elem, d_idx;
        int own;                // place of the row among the workgroup's own row dots
    };
    auto own_row0 = [&](int bq) __attribute__((always_inline)) -> int
    {
        return OWN ? (bq / p.n_batch - p.kv_group * hkv) * q_seq : 0;
    };
    auto query_rows = [&](int bq, int row0) __attribute__((always_inline)) -> QueryRows
    {
        if constexpr(GRID)
        {
            const int q_tile = (int)p.q_tile;
            const int tq = row0 / q_tile, t0 = tq * q_tile;
            const int64_t elem = (int64_t)bq * min(q_tile, q_seq - t0) + (row0 - t0);
            return QueryRows{p.Qt[q_tile0 + tq], p.dAt[q_tile0 + tq], p.lset[q_tile0 + tq], elem,
                d_slab + (int64_t)p.batch * t0 + elem, own_row0(bq) + row0};
        }
        else
        {
            const int64_t elem = (int64_t)bq * q_seq + row0;
            return QueryRows{p.Q, p.dA, p.lse, elem, elem, own_row0(bq) + row0};
        }
    };
    auto fetch_piece = [&](const QueryRows &at, bool at_end, char *qdst_base, char *gdst_base,
            int j) __attribute__((always_inline))
    {
        const char *Qp = static_cast<const char *>(at.Q) + at.elem * RB;
        const char *Gp = static_cast<const char *>(at.dA) + at.elem * RB;
        char *qdst = qdst_base + lds_grp + wave_u * LPW * 1024;
        char *gdst = gdst_base + lds_grp + wave_u * LPW * 1024;
        const uint32_t goff = at_end ? ld_goff_end[j] : ld_goff[j];
        load_to_lds16<0, false>(Qp, goff, qdst + j * 1024);
        load_to_lds16<0, false>(Gp, goff, gdst + j * 1024);
    };
    // (the same where the offsets are not kept; last: the step's last row that
    // exists, which the rows behind it read)
    auto fetch_piece_wide = [&](const QueryRows &at, int last, char *qdst_base, char *gdst_base,
            auto piece) __attribute__((always_inline))
    {
        constexpr int j = decltype(piece)::value;
        const char *Qp = static_cast<const char *>(at.Q) + at.elem * RB;
        const char *Gp = static_cast<const char *>(at.dA) + at.elem * RB;
        // (row wide_goff / RB + 4 * j of the step, or its last one: the offset is
        // not negative, the load widens it as unsigned)
        const uint32_t place = flip_bits<16 * j>(wide_goff);
        const int past = max((int)(place / (uint32_t)RB) + (4 * j - last), 0);
        const uint32_t goff = place + (uint32_t)((4 * j - past) * RB);
        load_to_lds16<0, false>(Qp, goff, qdst_base + lds_grp + wave_u * LPW * 1024 + j * 1024);
        load_to_lds16<0, false>(Gp, goff, gdst_base + lds_grp + wave_u * LPW * 1024 + j * 1024);
    };
    // The statistics of a step in two halves, so that the load's latency
    // passes behind the MFMAs of the step before: stat_load starts the read
    // of the lane's value (wavefront 0 a logsumexp, wavefront 1 a row dot),
    // stat_store turns it into what the step reads from LDS.
    auto stat_load = [&](const QueryRows &at, int last) __attribute__((always_inline)) -> float
    {
        float raw = 0.0f;
        // (in the wide body without a branch: the other wavefronts read along)
        if(OWN && wave_u == 1)
        {
            raw = DO_DK ? lds_own[at.own + min(lane, last)] : 0.0f;
        }
        else if(WIDE || wave_u < 2)
        {
            const float *src = wave_u % 2 == 0 ? at.lse + at.elem : p.D + at.d_idx;
            raw = src[min(WIDE ? lane_index_again() : lane, last)];
        }
        return raw;
    };
    auto stat_store = [&](float raw, int last, float (*stat)[kBwdStep])
        __attribute__((always_inline))
    {
        if(wave_u < 2)
        {
            const int r = WIDE ? lane_index_again() : lane;
            float v;
            if(wave_u == 0)
            {
                v = (r > last || raw == neg_inf()) ? __builtin_huge_valf() : raw * kLog2e;
            }
            else
            {
                v = r > last ? 0.0f : -raw;
            }
            stat[wave_u][r] = v;
        }
    };
    auto fetch_stat = [&](const QueryRows &at, int last, float (*stat)[kBwdStep])
    {
        stat_store(stat_load(at, last), last, stat);
    };
    constexpr int FETCH_STRIDE = (NNTILE_BWD_SPREAD == 2 ? NB : 1) * KSTEPS / LPW;
    static_assert(FETCH_STRIDE >= 1 && 1 + (LPW - 1) * FETCH_STRIDE < NB * KSTEPS,
            "the pieces of a fetch must fit between the MFMAs of a step");
    auto fetch = [&](int i, char *qdst_base, char *gdst_base, float (*stat)[kBwdStep])
    {
        int bq, qs;
        locate(i, bq, qs);
        const int row0 = qs * kBwdStep;
        const int last = min(kBwdStep, q_seq - row0) - 1;
        const QueryRows at = query_rows(bq, row0);
        if constexpr(WIDE)
        {
            each_slot([&](auto j) __attribute__((always_inline))
            {
                fetch_piece_wide(at, last, qdst_base, gdst_base, j);
            }, std::make_integer_sequence<int, LPW>{});
        }
        else if(LOADERS == kDkvWaves || wave_u < LOADERS)
        {
#pragma unroll
            for(int j = 0; j < LPW; ++j)
            {
                fetch_piece(at, last + 1 < kBwdStep, qdst_base, gdst_base, j);
            }
        }
        fetch_stat(at, last, stat);
    };

    // (the group's steps: every second of the walk)
    auto walk_own = [&](int i) __attribute__((always_inline)) -> int
    {
        const int n = walk_next(i);
        return GROUPS == 1 || n < 0 ? n : walk_next(n);
    };
    int i_cur = walk_begin(), i_last = -1;
    if(GROUPS > 1 && grp == 1 && i_cur >= 0)
    {
        i_last = -2;                        // (the first group has a step)
        i_cur = walk_next(i_cur);
    }
    if constexpr(OWN && DO_DK)
    {
        if(i_cur >= 0)
        {
            const QueryRows at = query_rows(nb + p.n_batch * (p.kv_group * hkv), 0);
            bwd_own_row_dots<T, HEAD>(static_cast<const uint16_t *>(at.dA) + at.elem * HEAD,
                    static_cast<const uint16_t *>(p.A) + at.elem * HEAD, p.kv_group * q_seq, q_seq,
                    (int64_t)(p.n_batch - 1) * q_seq * HEAD, lds_own);
            __syncthreads();
        }
    }
    if(i_cur >= 0)
    {
        fetch(i_cur, lds_q0, lds_g0, lds_stat[0]);
    }
    BWD_WALL_AT(3);     // (developer trace: the workgroup is set up, its first tile requested)
    auto step = [&](int i, int i_next, auto buf_tag, auto masked_tag)
        __attribute__((always_inline))
    {
        constexpr int BUF = decltype(buf_tag)::value;
        const char *Qs = BUF ? lds_q1 : lds_q0;
        const char *Gs = BUF ? lds_g1 : lds_g0;
        const float (*stat)[kBwdStep] = lds_stat[BUF];
        BWD_TRACE_START();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        BWD_TRACE_MARK(0);
        BWD_TRACE_STEP();
        // the statistics of the next step now, its tiles between the MFMAs
        // below (the last step loads its own tiles once more, rather than
        // branch)
        int bq_f, qs_f;
        locate(i_next >= 0 ? i_next : i, bq_f, qs_f);
        const int row0_f = qs_f * kBwdStep;
        const int last_f = min(kBwdStep, q_seq - row0_f) - 1;
        const bool at_end_f = last_f + 1 < kBwdStep;
        // (wave-common, computed once here: the loads between the MFMAs below
        // only add their offsets)
        const QueryRows at_f = query_rows(bq_f, row0_f);
        float raw_next = 0.0f;
        if(!WIDE && i_next >= 0)
        {
            raw_next = stat_load(at_f, last_f);
            if(NNTILE_BWD_SPREAD == 0 && (LOADERS == kDkvWaves || wave_u < LOADERS))
            {
#pragma unroll
                for(int j = 0; j < LPW; ++j)
                {
                    fetch_piece(at_f, at_end_f, BUF ? lds_q0 : lds_q1,
                            BUF ? lds_g0 : lds_g1, j);
                }
            }
        }
        int bq, qs;
        locate(i, bq, qs);
        constexpr bool use_mask = EXPLICIT && decltype(masked_tag)::value;
        const int q0 = qs * kBwdStep;
        const int rows_here = min(kBwdStep, q_seq - q0);
        // (wave-common: the workgroup's last key against the last key that
        // exists and the last key the step's first query sees)
        // (ruled: the mask of this step is the rule `key <= query + rel`)
        const bool ruled = MODE == NNTILE_HIP_MASK_CAUSAL
            || (EXPLICIT && !use_mask && !steps.is_open(qs));
        const bool bounds = k_row0 + ROWS > k_seq
            || (ruled && k_row0 + ROWS - 1 > rel + q0);
        const int vis_base = ruled ? rel + q0 : (1 << 30);
        // (the row stride through an empty asm statement: its multiples are
        // then computed where a step uses them - 32 scalar products - instead
        // of once before the loop and kept, which at head 128 means spilled)
        uint32_t mask_row_bytes = mask_row_bytes_wg;
        if(use_mask)
        {
            asm volatile("" : "+s"(mask_row_bytes));
        }
        const char *mask_step = static_cast<const char *>(p.mask)
            + (int64_t)q0 * (int64_t)mask_row_bytes;
        const uint32_t mask_last_row = (uint32_t)(rows_here - 1) * mask_row_bytes;

        if constexpr(WIDE)
        {
            // Both gradients at head 128: 192 registers hold fragments and
            // accumulators.  The step's two 32-query blocks go product by product,
            // S, dP, dV, dK, eight MFMAs each: 64 slots of one MFMA, the operand
            // read of the slot AHEAD later - across the products' borders - and a
            // slice of the vector work: P beside dP, dS beside dV.
            // Bound: the matrix pipe, 64 x 32 clocks a step and wavefront, at the
            // clock that the board's power leaves it (32 heads of 128, 4096 tokens,
            // causal, the whole call: 439 to 445 us with every MFMA behind its own
            // operand read, 435 to 437 so, on two boxes; the same bits.  Waves stood
            // at a wait or the barrier 43 % of their time, now 30 %, the matrix unit is
            // busy 65 % of the clocks for 60, of which there are 1.68 GHz for 1.79).
            static_assert(!use_mask, "masks given as values at head 128: dK and dV apart");
            constexpr int AHEAD = NNTILE_BWD_AHEAD_WIDE;
            constexpr int SLOTS = 64;
            enum { PART_S, PART_DP, PART_DV, PART_DK };
            f32x16 sv, dpv;
            uint32_t p_pk[8], ds_pk[8];
            vec8 ring[AHEAD + 1];
            f32x4 lse4;
            auto read = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                constexpr int mb = g / 32, part = g % 32 / 8, k = g % 8;
                if constexpr(g >= SLOTS)
                {
                    return;
                }
                else if constexpr(part == PART_S || part == PART_DP)
                {
                    ring[g % (AHEAD + 1)] = *reinterpret_cast<const vec8 *>(
                            (part == PART_S ? Qs : Gs) + mb * 32 * RB
                            + flip_bits<32 * k>(row_raddr[0]));
                }
                else
                {
                    constexpr int db = k / 2, t = 2 * mb + k % 2;
                    const char *src = (part == PART_DV ? Gs : Qs) + (16 * t) * RB;
                    const u32x2 lo = bwd_lds_read_tr16(src
                            + flip_bits<64 * db>(tr_raddr[0][0]));
                    const u32x2 hi = bwd_lds_read_tr16(src + 8 * RB
                            + flip_bits<64 * db + 32>(tr_raddr[0][0]));
                    const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                    ring[g % (AHEAD + 1)] = __builtin_bit_cast(vec8, raw);
                }
            };
            auto mfma = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                constexpr int part = g % 32 / 8, k = g % 8;
                const vec8 a = ring[g % (AHEAD + 1)];
                if constexpr(part == PART_S)
                {
                    sv = T::mfma(a, kf[k], k == 0 ? f32x16{} : sv);
                }
                else if constexpr(part == PART_DP)
                {
                    dpv = T::mfma(a, vf[k], dpv);
                }
                else
                {
                    constexpr int db = k / 2, tt = k % 2;
                    const uint32_t (&pk)[8] = part == PART_DV ? p_pk : ds_pk;
                    const u32x4 braw = {pk[4 * tt], pk[4 * tt + 1], pk[4 * tt + 2], pk[4 * tt + 3]};
                    f32x16 &to = part == PART_DV ? dv[db] : dk[db];
                    to = T::mfma(a, __builtin_bit_cast(vec8, braw), to);
                }
            };
            // the vector work beside slot g: the sixteen values of the product in
            // front, from the second slot on (the first is its last MFMA's time)
            auto vector_work = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                constexpr int mb = g / 32, part = g % 32 / 8, k = g % 8;
                if constexpr(part == PART_S && k < 4)
                {
                    // (dP - D: the accumulator starts at -D of its row)
                    const f32x4 nd4 = *reinterpret_cast<const f32x4 *>(
                            &stat[1][mb * 32 + 8 * k + 4 * half]);
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                    {
                        dpv[4 * k + e] = nd4[e];
                    }
                }
                // (values FIRST[k] .. FIRST[k + 1] beside slot k; of the logsumexps
                // four at a time have registers, read a slot ahead)
                constexpr int FIRST[9] = {0, 0, 2, 4, 6, 8, 12, 14, 16};
                if constexpr(part == PART_DP)
                {
#pragma unroll
                    for(int r = FIRST[k]; r < FIRST[k + 1]; ++r)
                    {
                        sv[r] = fast_exp2(fmaf(sv[r], c, -lse4[r % 4]));
                        if(r % 2 == 1)
                        {
                            p_pk[r / 2] = T::pack2(sv[r - 1], sv[r]);
                            asm volatile("" : "+v"(p_pk[r / 2]));
                        }
                    }
                    if constexpr(FIRST[k + 1] % 4 == 0 && k < 7)
                    {
                        lse4 = *reinterpret_cast<const f32x4 *>(
                                &stat[0][mb * 32 + 2 * FIRST[k + 1] + 4 * half]);
                    }
                }
                if constexpr(part == PART_DV)
                {
#pragma unroll
                    for(int r = FIRST[k]; r < FIRST[k + 1]; ++r)
                    {
                        dpv[r] = sv[r] * dpv[r];
                        if(r % 2 == 1)
                        {
                            ds_pk[r / 2] = T::pack2(dpv[r - 1], dpv[r]);
                            asm volatile("" : "+v"(ds_pk[r / 2]));
                        }
                    }
                }
            };
            each_slot(read, std::make_integer_sequence<int, AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            each_slot([&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if(g % 32 == 8 && bounds)
                {
                    // keys past the end and pairs the causal mask hides
                    float hidden = neg_inf();
                    asm volatile("" : "+v"(hidden));
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        // (the lane's part on the left, the rest is wave-common)
                        const int qr = g / 32 * 32 + tile_row(r, 0);
                        bool vis = k_ok;
                        if(MODE == NNTILE_HIP_MASK_CAUSAL)
                        {
                            vis = vis && (my_k_less_half <= vis_base + qr);
                        }
                        sv[r] = vis ? sv[r] : hidden;
                    }
                }
                read(std::integral_constant<int, g + AHEAD>{});
                mfma(slot);
                vector_work(slot);
                // the next step's rows early in the step, its statistics half way
                if constexpr(g % 8 == 2 && g / 8 < LPW)
                {
                    fetch_piece_wide(at_f, last_f, BUF ? lds_q0 : lds_q1, BUF ? lds_g0 : lds_g1,
                            std::integral_constant<int, g / 8>{});
                }
                if constexpr(g == SLOTS / 2)
                {
                    raw_next = stat_load(at_f, last_f);
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, SLOTS>{});
        }
        else if constexpr(use_mask || NNTILE_BWD_PIPE == 0)
        {
            // (one 32-query block at a time: half the accumulators live)
            // ---- S = Q K^T, dP = dA V^T: rows are queries, the lane's column its key;
            // P, dS: register r of block mb is query q0 + mb*32 + tile_row(r, half) --------------
#pragma unroll
            for(int mb = 0; mb < NB; ++mb)
            {
                uint32_t p_pk[8], ds_pk[8];
                f32x16 sv, dpv;
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    sv[r] = 0.0f;
                    dpv[r] = 0.0f;
                }
                if(DO_DK)
                {
                    // dP - D: the accumulator starts at -D of its row (four
                    // consecutive queries per LDS read), the products add dP
#pragma unroll
                    for(int rg = 0; rg < 4; ++rg)
                    {
                        const f32x4 nd4 = *reinterpret_cast<const f32x4 *>(
                                &stat[1][(mb + kh) * 32 + 8 * rg + 4 * half]);
#pragma unroll
                        for(int e = 0; e < 4; ++e)
                        {
                            dpv[4 * rg + e] = nd4[e];
                        }
                    }
                }
#pragma unroll
                for(int ks = 0; ks < KSTEPS; ++ks)
                {
                    const vec8 qa = *reinterpret_cast<const vec8 *>(Qs + row_raddr[ks] + mb * 32 * RB);
                    sv = T::mfma(qa, kf[ks], sv);
                    if(DO_DK)
                    {
                        const vec8 ga = *reinterpret_cast<const vec8 *>(Gs + row_raddr[ks]
                                + mb * 32 * RB);
                        dpv = T::mfma(ga, vf[ks], dpv);
                    }
                    if(LOADERS == kDkvWaves || wave_u < LOADERS)
                    {
#pragma unroll
                        for(int j = 0; j < LPW; ++j)
                        {
                            if(NNTILE_BWD_SPREAD != 0 && mb * KSTEPS + ks == 1 + j * FETCH_STRIDE)
                            {
                                fetch_piece(at_f, at_end_f, BUF ? lds_q0 : lds_q1,
                                        BUF ? lds_g0 : lds_g1, j);
                            }
                        }
                    }
                }
                // Keys past the end and pairs the causal mask hides: their scores
                // become -inf in a pass of their own, which only the workgroups at
                // the end of the keys and the steps on the diagonal run (a
                // wave-common branch).
                if(bounds)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        // (the lane's part on the left, the rest is wave-common)
                        const int qr = mb * 32 + tile_row(r, 0);
                        bool vis = k_ok;
                        if(MODE == NNTILE_HIP_MASK_CAUSAL || EXPLICIT)
                        {
                            vis = vis && (my_k_less_half <= vis_base + qr);
                        }
                        sv[r] = vis ? sv[r] : neg_inf();
                    }
                }
                float pv[16], dsv[16];
#pragma unroll
                for(int rg = 0; rg < 4; ++rg)
                {
                    // four consecutive queries: their statistics in one LDS read each
                    const int qr0 = (mb + kh) * 32 + 8 * rg + 4 * half;
                    const f32x4 lse4 = *reinterpret_cast<const f32x4 *>(&stat[0][qr0]);
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                    {
                        const int r = 4 * rg + e;
                        float ex = fmaf(sv[r], c, -lse4[e]);    // -inf: hidden, or a row past the end
                        bool visible = true;
                        if(use_mask)
                        {
                            // the row is the same for the lanes of one half: its
                            // address is wave-common, the lane adds its key (and
                            // four rows in the upper half, while those exist;
                            // rows past the end read a row that exists and are
                            // dropped by their logsumexp of +inf)
                            const int rb = (mb + kh) * 32 + 8 * rg + e;
                            const char *mrow = mask_step
                                + min((uint32_t)rb * mask_row_bytes, mask_last_row);
                            const char *mp = mrow + (rb + 4 < rows_here ? mask_off_hi : mask_off_lo);
                            if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                            {
                                const float add = T::to_float(
                                        *reinterpret_cast<const uint16_t *>(mp));
                                visible = visible && (add != neg_inf());
                                ex = fmaf(add, kLog2e, ex);
                            }
                            else
                            {
                                const uint8_t shown = *reinterpret_cast<const uint8_t *>(mp);
                            visible = visible && (shown != 0);
                            }
                        }
                        pv[r] = use_mask ? (visible ? fast_exp2(ex) : 0.0f) : fast_exp2(ex);
                        dsv[r] = pv[r] * dpv[r];
                    }
                }
#pragma unroll
                for(int k = 0; k < 8; ++k)
                {
                    p_pk[k] = T::pack2(pv[2 * k], pv[2 * k + 1]);
                    ds_pk[k] = T::pack2(dsv[2 * k], dsv[2 * k + 1]);
                }
                // ---- dV^T += dA^T P, dK^T += Q^T dS: the block's two sub-steps of 16 queries ----
#pragma unroll
                for(int tt = 0; tt < 2; ++tt)
                {
                    const int t = 2 * mb + tt;
                    const u32x4 praw = {p_pk[4 * tt], p_pk[4 * tt + 1], p_pk[4 * tt + 2],
                        p_pk[4 * tt + 3]};
                    const u32x4 sraw = {ds_pk[4 * tt], ds_pk[4 * tt + 1], ds_pk[4 * tt + 2],
                        ds_pk[4 * tt + 3]};
                    const vec8 pb = __builtin_bit_cast(vec8, praw);
                    const vec8 sb = __builtin_bit_cast(vec8, sraw);
#pragma unroll
                    for(int db = 0; db < DBLOCKS; ++db)
                    {
                        if(DO_DV)
                        {
                            const u32x2 glo = bwd_lds_read_tr16(Gs + tr_raddr[0][db] + (16 * t) * RB);
                            const u32x2 ghi = bwd_lds_read_tr16(Gs + tr_raddr[1][db] + (16 * t) * RB);
                            const u32x4 graw = {glo[0], glo[1], ghi[0], ghi[1]};
                            dv[db] = T::mfma(__builtin_bit_cast(vec8, graw), pb, dv[db]);
                        }
                        if(DO_DK)
                        {
                            const u32x2 qlo = bwd_lds_read_tr16(Qs + tr_raddr[0][db] + (16 * t) * RB);
                            const u32x2 qhi = bwd_lds_read_tr16(Qs + tr_raddr[1][db] + (16 * t) * RB);
                            const u32x4 qraw = {qlo[0], qlo[1], qhi[0], qhi[1]};
                            dk[db] = T::mfma(__builtin_bit_cast(vec8, qraw), sb, dk[db]);
                        }
                    }
                }
            }
        }
        else if constexpr(KH > 1)
        {
            // One block of 32 queries: S, dP with P beside it, dV^T += dA^T P with dS
            // beside it, dK^T += Q^T dS - those of them that this part has - in slots
            // as below.
            f32x16 sv, dpv;
            uint32_t p_pk[8], ds_pk[8];
            constexpr int N_DP = DO_DK ? KSTEPS : 0, N_DV = DO_DV ? 2 * DBLOCKS : 0;
            constexpr int AT_DV = KSTEPS + N_DP, AT_DK = AT_DV + N_DV;
            constexpr int SLOTS = AT_DK + (DO_DK ? 2 * DBLOCKS : 0);
            constexpr int AHEAD = kBwdAhead<HEAD>;
            vec8 ring[AHEAD + 1];
            auto read = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g < AT_DV)
                {
                    ring[g % (AHEAD + 1)] = *reinterpret_cast<const vec8 *>((g < KSTEPS ? Qs : Gs)
                            + row_raddr[g % KSTEPS]);
                }
                else if constexpr(g < SLOTS)
                {
                    constexpr int i = g < AT_DK ? g - AT_DV : g - AT_DK;
                    constexpr int t = i / DBLOCKS, db = i % DBLOCKS;
                    const char *src = (g < AT_DK ? Gs : Qs) + (16 * t) * RB;
                    const u32x2 lo = bwd_lds_read_tr16(src + tr_raddr[0][db]);
                    const u32x2 hi = bwd_lds_read_tr16(src + tr_raddr[1][db]);
                    const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                    ring[g % (AHEAD + 1)] = __builtin_bit_cast(vec8, raw);
                }
            };
            auto four = [&](int which, int rg) __attribute__((always_inline)) -> f32x4
            {
                return *reinterpret_cast<const f32x4 *>(&stat[which][kh * 32 + 8 * rg + 4 * half]);
            };
            f32x4 lse4[4];
            // probabilities [first, last) of the block
            auto p_items = [&](int first, int last) __attribute__((always_inline))
            {
#pragma unroll
                for(int r = first; r < last; ++r)
                {
                    sv[r] = fast_exp2(fmaf(sv[r], c, -lse4[r / 4][r % 4]));
                    if(DO_DV && r % 2 == 1)
                    {
                        p_pk[r / 2] = T::pack2(sv[r - 1], sv[r]);
                    }
                }
            };
            auto ds_items = [&](int first, int last) __attribute__((always_inline))
            {
#pragma unroll
                for(int r = first; r < last; ++r)
                {
                    dpv[r] = sv[r] * dpv[r];
                    if(r % 2 == 1)
                    {
                        ds_pk[r / 2] = T::pack2(dpv[r - 1], dpv[r]);
                    }
                }
            };
            each_slot(read, std::make_integer_sequence<int, AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            each_slot([&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g == KSTEPS)
                {
                    // (keys past the end and pairs the rule hides: see below)
                    if(bounds)
                    {
#pragma unroll
                        for(int r = 0; r < 16; ++r)
                        {
                            bool vis = k_ok;
                            if(MODE == NNTILE_HIP_MASK_CAUSAL || EXPLICIT)
                            {
                                vis = vis && (my_k_less_half <= vis_base + tile_row(r, 0));
                            }
                            sv[r] = vis ? sv[r] : neg_inf();
                        }
                    }
                    if constexpr(!DO_DK)
                    {
                        p_items(0, 16);
                    }
                }
                if constexpr(DO_DK && !DO_DV && g == AT_DK)
                {
                    ds_items(0, 16);
                }
                read(std::integral_constant<int, g + AHEAD>{});
                const vec8 a = ring[g % (AHEAD + 1)];
                if constexpr(g < KSTEPS)
                {
                    sv = T::mfma(a, kf[g], g == 0 ? f32x16{} : sv);
                    if(LOADERS == kDkvWaves || wave_u < LOADERS)
                    {
#pragma unroll
                        for(int j = 0; j < LPW; ++j)
                        {
                            if(NNTILE_BWD_SPREAD != 0 && g == 1 + j * FETCH_STRIDE)
                            {
                                fetch_piece(at_f, at_end_f, BUF ? lds_q0 : lds_q1,
                                        BUF ? lds_g0 : lds_g1, j);
                            }
                        }
                    }
                    // the statistics of the rows, over the first slots
#pragma unroll
                    for(int rg = g * 4 / KSTEPS; rg < (g + 1) * 4 / KSTEPS; ++rg)
                    {
                        lse4[rg] = four(0, rg);
                        if(DO_DK)
                        {
                            // dP - D: the accumulator starts at -D of its row
                            const f32x4 nd4 = four(1, rg);
#pragma unroll
                            for(int e = 0; e < 4; ++e)
                            {
                                dpv[4 * rg + e] = nd4[e];
                            }
                        }
                    }
                }
                else if constexpr(g < AT_DV)
                {
                    constexpr int i = g - KSTEPS;
                    dpv = T::mfma(a, vf[i], dpv);
                    p_items(i * 16 / KSTEPS, (i + 1) * 16 / KSTEPS);
                }
                else if constexpr(g < AT_DK)
                {
                    constexpr int i = g - AT_DV, t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x4 braw = {p_pk[4 * t], p_pk[4 * t + 1], p_pk[4 * t + 2], p_pk[4 * t + 3]};
                    dv[db] = T::mfma(a, __builtin_bit_cast(vec8, braw), dv[db]);
                    if constexpr(BOTH)
                    {
                        ds_items(i * 16 / N_DV, (i + 1) * 16 / N_DV);
                    }
                }
                else
                {
                    constexpr int i = g - AT_DK, t = i / DBLOCKS, db = i % DBLOCKS;
                    const u32x4 braw = {ds_pk[4 * t], ds_pk[4 * t + 1], ds_pk[4 * t + 2],
                        ds_pk[4 * t + 3]};
                    dk[db] = T::mfma(a, __builtin_bit_cast(vec8, braw), dk[db]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, SLOTS>{});
        }
        else
        {
            // The step's two 32-query blocks in three phases each - A: S = Q K^T and
            // dP = dA V^T (rows are queries, the lane's column its key), B: P and dS
            // on the vector ALU, C: dV^T += dA^T P, dK^T += Q^T dS - issued as
            // A0 | A1 with B0 | C0 with B1 | C1, so that the matrix unit works
            // through a block's neighbours while the vector ALU turns its scores
            // into probabilities.  P, dS: register r of block mb is query
            // q0 + mb*32 + tile_row(r, half).
            f32x16 sv[2], dpv[2];
            uint32_t p_pk[2][8], ds_pk[2][8];
            // Keys past the end and pairs the causal mask hides: their scores
            // become -inf in a pass of their own, which only the workgroups at
            // the end of the keys and the steps on the diagonal run (a
            // wave-common branch).
            auto hide = [&](int mb) __attribute__((always_inline))
            {
                if(bounds)
                {
#pragma unroll
                    for(int r = 0; r < 16; ++r)
                    {
                        // (the lane's part on the left, the rest is wave-common)
                        const int qr = mb * 32 + tile_row(r, 0);
                        bool vis = k_ok;
                        if(MODE == NNTILE_HIP_MASK_CAUSAL || EXPLICIT)
                        {
                            vis = vis && (my_k_less_half <= vis_base + qr);
                        }
                        sv[mb][r] = vis ? sv[mb][r] : neg_inf();
                    }
                }
            };
            // The overlapped order, written out slot by slot (one MFMA, the operand
            // read of the slot AHEAD later - of the next phase too -, a slice of the
            // vector work) with a scheduling barrier after each, or the compiler
            // regroups it into phases.
            constexpr int A_MFMAS = (DO_DK ? 2 : 1) * KSTEPS, C_MFMAS = (BOTH ? 2 : 1) * 2 * DBLOCKS;
            constexpr int SLOTS = 2 * (A_MFMAS + C_MFMAS);
            constexpr int AHEAD = kBwdAhead<HEAD>;
            vec8 ring[AHEAD + 1];
            auto read = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                if constexpr(g < 2 * A_MFMAS)
                {
                    constexpr int mb = g / A_MFMAS, i = g % A_MFMAS, ks = DO_DK ? i / 2 : i;
                    const char *src = (DO_DK && (i & 1)) ? Gs : Qs;
                    ring[g % (AHEAD + 1)] = *reinterpret_cast<const vec8 *>(src + row_raddr[ks]
                            + mb * 32 * RB);
                }
                else if constexpr(g < SLOTS)
                {
                    // (both gradients: dV and dK products alternate)
                    constexpr int i = (g - 2 * A_MFMAS) % C_MFMAS, mb = (g - 2 * A_MFMAS) / C_MFMAS;
                    constexpr int j = BOTH ? i / 2 : i;
                    constexpr bool for_dv = BOTH ? (i & 1) == 0 : DO_DV;
                    constexpr int t = 2 * mb + j / DBLOCKS, db = j % DBLOCKS;
                    const char *src = (for_dv ? Gs : Qs) + (16 * t) * RB;
                    const u32x2 lo = bwd_lds_read_tr16(src + tr_raddr[0][db]);
                    const u32x2 hi = bwd_lds_read_tr16(src + tr_raddr[1][db]);
                    const u32x4 raw = {lo[0], lo[1], hi[0], hi[1]};
                    ring[g % (AHEAD + 1)] = __builtin_bit_cast(vec8, raw);
                }
            };
            auto mfma = [&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                const vec8 a = ring[g % (AHEAD + 1)];
                if constexpr(g < 2 * A_MFMAS)
                {
                    constexpr int mb = g / A_MFMAS, i = g % A_MFMAS, ks = DO_DK ? i / 2 : i;
                    if constexpr(DO_DK && (i & 1))
                    {
                        dpv[mb] = T::mfma(a, vf[ks], dpv[mb]);
                    }
                    else
                    {
                        sv[mb] = T::mfma(a, kf[ks], ks == 0 ? f32x16{} : sv[mb]);
                    }
                    // the tile loads of the next step, spread over the products
                    if((LOADERS == kDkvWaves || wave_u < LOADERS) && NNTILE_BWD_SPREAD != 0
                            && (!DO_DK || (i & 1)))
                    {
#pragma unroll
                        for(int j = 0; j < LPW; ++j)
                        {
                            if(mb * KSTEPS + ks == 1 + j * FETCH_STRIDE)
                            {
                                fetch_piece(at_f, at_end_f, BUF ? lds_q0 : lds_q1,
                                        BUF ? lds_g0 : lds_g1, j);
                            }
                        }
                    }
                }
                else
                {
                    constexpr int i = (g - 2 * A_MFMAS) % C_MFMAS, mb = (g - 2 * A_MFMAS) / C_MFMAS;
                    constexpr int j = BOTH ? i / 2 : i;
                    constexpr bool for_dv = BOTH ? (i & 1) == 0 : DO_DV;
                    constexpr int tt = j / DBLOCKS, db = j % DBLOCKS;
                    const uint32_t (&pk)[8] = for_dv ? p_pk[mb] : ds_pk[mb];
                    const u32x4 braw = {pk[4 * tt], pk[4 * tt + 1], pk[4 * tt + 2], pk[4 * tt + 3]};
                    f32x16 &to = for_dv ? dv[db] : dk[db];
                    to = T::mfma(a, __builtin_bit_cast(vec8, braw), to);
                }
            };
            auto a_init = [&](int mb) __attribute__((always_inline))
            {
                if(DO_DK)
                {
#pragma unroll
                    for(int rg = 0; rg < 4; ++rg)
                    {
                        const f32x4 nd4 = *reinterpret_cast<const f32x4 *>(
                                &stat[1][mb * 32 + 8 * rg + 4 * half]);
#pragma unroll
                        for(int e = 0; e < 4; ++e)
                        {
                            dpv[mb][4 * rg + e] = nd4[e];
                        }
                    }
                }
            };
            // vector work of query r of block mb (statistics of four queries per
            // LDS read, read one group ahead)
            f32x4 lse_cur = {0.0f, 0.0f, 0.0f, 0.0f}, lse_nxt = lse_cur;
            float pv_even = 0.0f, ds_even = 0.0f;
            auto b_begin = [&](int mb) __attribute__((always_inline))
            {
                lse_nxt = *reinterpret_cast<const f32x4 *>(&stat[0][mb * 32 + 4 * half]);
            };
            // (in three stages a tick apart - exponent, exponential, products and
            // packing - so that a lone wavefront does not wait for its own
            // results: tick t takes query t, t-1 and t-2 through one stage each)
            float ex_stage[2] = {0.0f, 0.0f}, pr_stage[2] = {0.0f, 0.0f};
            auto b_tick = [&](int mb, int t) __attribute__((always_inline))
            {
                if(t - 2 >= 0 && t - 2 < 16)
                {
                    const int r = t - 2;
                    const float pr = pr_stage[r % 2];
                    const float dsr = pr * dpv[mb][r];
                    if(r % 2 == 0)
                    {
                        pv_even = pr;
                        ds_even = dsr;
                    }
                    else
                    {
                        if(DO_DV)
                        {
                            p_pk[mb][r / 2] = T::pack2(pv_even, pr);
                            asm volatile("" : "+v"(p_pk[mb][r / 2]));
                        }
                        if(DO_DK)
                        {
                            ds_pk[mb][r / 2] = T::pack2(ds_even, dsr);
                            asm volatile("" : "+v"(ds_pk[mb][r / 2]));
                        }
                    }
                }
                if(t - 1 >= 0 && t - 1 < 16)
                {
                    const int r = t - 1;
                    pr_stage[r % 2] = fast_exp2(ex_stage[r % 2]);
                }
                if(t < 16)
                {
                    const int r = t;
                    if(r % 4 == 0)
                    {
                        lse_cur = lse_nxt;
                        if(r + 4 < 16)
                        {
                            lse_nxt = *reinterpret_cast<const f32x4 *>(
                                    &stat[0][mb * 32 + 8 * (r / 4 + 1) + 4 * half]);
                        }
                    }
                    ex_stage[r % 2] = fmaf(sv[mb][r], c, -lse_cur[r % 4]);
                }
            };
            constexpr int B_TICKS = 18;
            a_init(0);
            each_slot(read, std::make_integer_sequence<int, AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            each_slot([&](auto slot) __attribute__((always_inline))
            {
                constexpr int g = decltype(slot)::value;
                constexpr int i1 = g - A_MFMAS, i2 = g - 2 * A_MFMAS;
                // (the second block's start and the first's statistics ahead of the
                // phase that needs them)
                if constexpr(g == A_MFMAS - 1)
                {
                    a_init(1);
                    b_begin(0);
                }
                if constexpr(i1 == 0)
                {
                    BWD_TRACE_MARK(1);
                    hide(0);
                }
                if constexpr(i2 == 0)
                {
                    BWD_TRACE_MARK(2);
                    hide(1);
                    b_begin(1);
                }
                if constexpr(i2 == C_MFMAS)
                {
                    BWD_TRACE_MARK(3);
                }
                read(std::integral_constant<int, g + AHEAD>{});
                mfma(slot);
                if constexpr(i1 >= 0 && i1 < A_MFMAS)
                {
#pragma unroll
                    for(int t = i1 * B_TICKS / A_MFMAS; t < (i1 + 1) * B_TICKS / A_MFMAS; ++t)
                    {
                        b_tick(0, t);
                    }
                }
                if constexpr(i2 >= 0 && i2 < C_MFMAS)
                {
#pragma unroll
                    for(int t = i2 * B_TICKS / C_MFMAS; t < (i2 + 1) * B_TICKS / C_MFMAS; ++t)
                    {
                        b_tick(1, t);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, SLOTS>{});
        }
        BWD_TRACE_MARK(4);
        // (the other buffer's readers passed this step's barrier; the next
        // step's barrier orders these writes before its reads)
        __builtin_amdgcn_sched_barrier(0);
        if(i_next >= 0)
        {
            stat_store(raw_next, last_f, lds_stat[BUF ^ 1]);
        }
        BWD_TRACE_MARK(5);
    };
    auto run = [&](int i, int i_next, auto buf_tag) __attribute__((always_inline))
    {
        if(EXPLICIT && !steps.is_open(i % kHeadStride) && !steps.is_rule(i % kHeadStride))
        {
            step(i, i_next, buf_tag, std::true_type{});
        }
        else
        {
            step(i, i_next, buf_tag, std::false_type{});
        }
    };
    while(i_cur >= 0)
    {
        int i_next = walk_own(i_cur);
        run(i_cur, i_next, std::integral_constant<int, 0>{});
        i_last = i_cur;
        i_cur = i_next;
        if(i_cur < 0)
        {
            break;
        }
        i_next = walk_own(i_cur);
        run(i_cur, i_next, std::integral_constant<int, 1>{});
        i_last = i_cur;
        i_cur = i_next;
    }
    // (the last step's spare loads into LDS must have landed before the
    // workgroup's LDS can be given away)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // (one barrier a step: the second group meets that of a last step it has not)
    if(GROUPS > 1 && grp == 1 && (i_last == -2 || (i_last >= 0 && walk_next(i_last) >= 0)))
    {
        __syncthreads();
    }

    BWD_TRACE_FLUSH(PART);
    // ---- dK (+)= scale dk, dV (+)= dv (every wavefront is done with the tiles in LDS) ---
    __syncthreads();
    const int row_first = k_row0 + rows32 * 32;
    char *xch = (wave_u == 0 ? lds_q0 : wave_u == 1 ? lds_q1 : wave_u == 2 ? lds_g0 : lds_g1) + lds_grp;
    if constexpr(GROUPS > 1)
    {
        static_assert(BOTH, "two groups: both gradients in one workgroup");
        bwd_add_groups<DBLOCKS, G::BYTES>(grp, xch, dk);
        __syncthreads();            // (the first sums have been read)
        bwd_add_groups<DBLOCKS, G::BYTES>(grp, xch, dv);
        if(grp == 1)
        {
            return;
        }
    }
    const int64_t first_byte = row_elem(row_first, true) * RB + kh * (RB / 2);
    const char *other = wave_u == 0 ? lds_g0 : wave_u == 1 ? lds_g1 : wave_u == 2 ? lds_q0 : lds_q1;
    char *rows = KH > 1 ? xch + G::BYTES - 32 * (RB / 2) : xch;     // (behind the sums handed over)
    if constexpr(KH > 1 && DO_DK)
    {
        bwd_add_halves<DBLOCKS / 2>(xch, other, dk);
    }
    if(DO_DK)
    {
        bwd_store_rows<T, HEAD, KH>(rows, static_cast<char *>(dK_own) + first_byte, k_seq - row_first,
                dk, p.scale, !p.overwrite);
    }
    if constexpr(KH > 1 && DO_DV)
    {
        if(BOTH)
        {
            __syncthreads();        // (the first sums have been read)
        }
        bwd_add_halves<DBLOCKS / 2>(xch, other, dv);
    }
    if(DO_DV)
    {
        bwd_store_rows<T, HEAD, KH>(rows, static_cast<char *>(dV_own) + first_byte, k_seq - row_first,
                dv, 1.0f, !p.overwrite);
    }
}

// One launch for the three gradients: workgroups [0, n_dkv) compute dK,
// the next n_dq dQ (three products a step each, the longer workgroups), the
// last n_dkv dV.  A tile-pair call has fewer workgroups per gradient than the
// chip has places (two a CU); together they fill it, and a long call loses
// the ends of two launches.
template<typename T, int HEAD, int MODE, bool GRID, bool FUSED_KEYS = false, int GROUPS = 1, int KH = 1,
        bool OWN = false>
__global__ __launch_bounds__(kDkvThreads * GROUPS, 2)
void sdpa_bwd_kernel(const std::conditional_t<GRID, BwdGridParams, BwdParams> p, unsigned n_dkv,
        unsigned n_dq)
{
    BWD_WALL(0, blockIdx.x < n_dkv ? 1 : (blockIdx.x < n_dkv + n_dq ? 0 : 2));
    typedef BwdTile<HEAD> G;
    static_assert(kDkvThreads == kBwdThreads, "one block size for the three parts");
    __shared__ __attribute__((aligned(1024))) char lds_0[G::BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_1[G::BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_2[G::BYTES * GROUPS];
    __shared__ __attribute__((aligned(1024))) char lds_3[G::BYTES * GROUPS];
    // dK, dV parts, per query of a step: logsumexp in log2 units (+inf for a
    // row that saw nothing) and minus the row dot D; rows past the end hold +inf / 0
    __shared__ __attribute__((aligned(16))) float lds_stat_all[GROUPS][2][2][kBwdStep];
    __shared__ float lds_own[OWN ? kBwdOwnRows : 1];
    __shared__ uint32_t lds_word;
    if constexpr(OWN)
    {
        lds_word = 0u;
        __syncthreads();
    }
    const int grp = GROUPS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kDkvThreads) : 0;
    float (*const lds_stat)[2][kBwdStep] = lds_stat_all[grp];
    if constexpr(FUSED_KEYS)
    {
        // (K and V fragments and both accumulators fit beside the rest: one
        // set of key-owning workgroups computes dK and dV from one pass over
        // the scores, seven products a call instead of eight)
        if(blockIdx.x < n_dkv)
        {
            sdpa_bwd_dkv_body<T, HEAD, MODE, BWD_PART_DK | BWD_PART_DV, GRID, GROUPS, KH, OWN>(p, blockIdx.x, lds_0,
                    lds_1, lds_2, lds_3, lds_stat, &lds_word, lds_own);
        }
        else
        {
            sdpa_bwd_dq_body<T, HEAD, MODE, GRID, GROUPS, KH, OWN>(p, blockIdx.x - n_dkv, lds_0, lds_1, lds_2, lds_3, &lds_word);
        }
    }
    else if(blockIdx.x < n_dkv)
    {
        sdpa_bwd_dkv_body<T, HEAD, MODE, BWD_PART_DK, GRID, GROUPS, KH, OWN>(p, blockIdx.x, lds_0, lds_1, lds_2,
                lds_3, lds_stat, &lds_word, lds_own);
    }
    else if(blockIdx.x < n_dkv + n_dq)
    {
        sdpa_bwd_dq_body<T, HEAD, MODE, GRID, GROUPS, KH, OWN>(p, blockIdx.x - n_dkv, lds_0, lds_1, lds_2, lds_3, &lds_word);
    }
    else
    {
        sdpa_bwd_dkv_body<T, HEAD, MODE, BWD_PART_DV, GRID, GROUPS, KH, OWN>(p, blockIdx.x - n_dkv - n_dq, lds_0,
                lds_1, lds_2, lds_3, lds_stat, &lds_word, lds_own);
    }
#ifdef NNTILE_BWD_TRACE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    BWD_WALL(1, blockIdx.x < n_dkv ? 1 : (blockIdx.x < n_dkv + n_dq ? 0 : 2));
#endif
}

static BwdPreludeParams prelude_params(const BwdParams &p, int64_t q_tile, int n_q_tiles)
{
    BwdPreludeParams pre = {};
    pre.q_seq = p.q_seq;
    pre.q_tile = q_tile;
    pre.mask_ld = p.mask_ld;
    pre.D = p.D;
    pre.mask = p.mask;
    pre.k_seq = (int32_t)p.k_seq;
    pre.batch = p.batch;
    pre.n_q_tiles = n_q_tiles;
    return pre;
}

template<typename T, int HEAD, int MODE>
static int launch_prelude(hipStream_t stream, BwdPreludeParams &pre, int n_tiles)
{
    constexpr int ROWS = 256 / (HEAD / 8) * kRowdotRows;
    const int64_t rows = (int64_t)pre.batch * (pre.q_tile < pre.q_seq ? pre.q_tile : pre.q_seq);
    const int64_t per_tile = (rows + ROWS - 1) / ROWS;
    const int64_t n_wgs = pre.n_class_wgs + per_tile * n_tiles;
    if(per_tile > 0x7fffffff || n_wgs > 0x7fffffff)
    {
        return NNTILE_HIP_EINVAL;
    }
    pre.wgs_per_tile = (int32_t)per_tile;
    hipLaunchKernelGGL((sdpa_bwd_prelude_kernel<T, HEAD, MODE == NNTILE_HIP_MASK_CAUSAL
                ? NNTILE_HIP_MASK_NONE : MODE>), dim3((unsigned)n_wgs), dim3(256), 0, stream, pre);
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

// Steps of the longest walk - the queries of all heads of a group, or the keys - from which
// it is a long one
constexpr int64_t kBwdLongWalk = 13;
static int64_t bwd_longest_walk(const BwdParams &p)
{
    const int64_t keys = (p.k_seq + kBwdStep - 1) / kBwdStep;
    const int64_t queries = (p.q_seq + kBwdStep - 1) / kBwdStep * p.kv_group;
    return keys > queries ? keys : queries;
}

// Workgroups of 64 rows whose wavefronts halve the steps of the walk between them
// (sdpa_bwd_kernel, KH == 2): launches that leave CUs empty or with one wavefront on each
// SIMD, waiting for its own operands, have twice the workgroups so with half of the chain
// each, and skip blocks of a mask for 64 rows instead of 128; a launch that fills the chip
// loses by it, as every step comes into LDS twice as often for its MFMAs (32 x 4096 of head
// 128, causal, 463 / 594 us).
//
// The rule, in workgroups of 64 rows, dK and dV apart / together in one (head 64; at head
// 128 that does not fit the registers):
//   masks as values     apart up to two a CU, else together up to two
//   a rule, head 64     apart up to one a CU, else together up to four (open: two), or where
//                       a group's heads make the key blocks' walks the longest: 256 (208) of them
//   a rule, head 128    apart up to three a CU (open: two), or 256 (128) of grouped heads
// but for two lines that are not there for speed: launches on either side of them give
// equal bits, which tests of this repository hold them to (the calls over slabs of 12
// heads of 1024 rows in test_gpu_backward_grid.py, the rectangular ones of
// test_gpu_backward_wide_keys.py), although a call's last bit may otherwise depend on
// what shares its launch (head 64, causal, whole / halved: 12 x 1024 23.8 / -, beside it 16 x
// 1000 26.5 / 20.8).
//
// Whole calls, us, fp16, before / apart / together:
//   masks as values, head 64: 2 x 128 10.9 / 8.9 / 10.3, 12 x 500 causal 18.1 / 14.8 / 16.7,
//     open 18.7 / 18.2 / 18.0, a window 18.2 / 13.8 / 17.7; 8 x 1000 25.3 / 23.7 / 23.9, 27.3 /
//     26.9 / 26.4, 19.0 / 14.7 / 18.9; 32 x 500 24.1 / 22.2 / 19.9, 26.1 / 24.4 / 21.9, 25.0 / 18.7 /
//     21.5; 24 x 1000 36.0 / 34.8 / 30.8, 41.0 / 51.4 / 45.7, 43.5 / 27.1 / 32.2: not;
//   head 128: 4 x 500 22.8 / 17.7, 25.0 / 19.0, 29.5 / 18.4; 8 x 1000 37.3 / 31.5, 42.0 / 36.8, 34.4 /
//     24.5; 24 x 500 28.4 / 25.4, 32.2 / 34.8, 38.4 / 33.3: not;
//   a rule, head 64: 4 x 1000 19.5 / 16.7 / 18.4, open 20.6 / 18.0 / 18.8, 8 x 1000 20.6 / 20.0 / 18.9,
//     21.4 / 20.8 / 19.5; 16 x 1000 27.5 / 25.4 / 22.0, 29.8 / 29.0 / 25.0; 24 x 1000 28.6 / 30.3 / 26.2,
//     34.8 / 42.8 / 40.2; 16 x 2000 47.3 / 55.4 / 45.7; 64 x 1000 47.8 / 59.8 / 53.4;
//   head 128: 8 x 500 19.6 / 15.5, open 19.1 / 15.6, 8 x 1000 28.9 / 26.1, 29.9 / 29.1, 16 x 1000 38.6 /
//     35.0, 44.3 / 48.0, 4 x 4000 113 / 87, 24 x 1000 43.5 / 45.1;
//   grouped heads, whose longest chain is a key block's walk over all queries of its group:
//     head 64, 32 on 8 x 1500 89.9 / 89.9 / 78.9, open 95.2 / 123 / 88.7, 64 on 16 x 800 54.5 / 56.4 /
//     48.4, 59.6 / 76.3 / 54.0, x 2500 open 384 / 504 / 413; head 128, 32 on 8 x 800 80.7 / 55.6, 92.2 /
//     66.6, x 1500 153 / 126, 169 / 180, 16 on 2 x 4000 728 / 526, 788 / 670; 32 on 16 x 900 57.3 /
//     59.1.
enum { BWD_WHOLE_STEPS, BWD_HALVED_APART, BWD_HALVED_BOTH };
static int bwd_halved(const BwdParams &p, int head, int mode, int64_t entries, int64_t n_dkv,
        int64_t n_dq)
{
    const int64_t apart = 2 * n_dkv + n_dq, both = n_dkv + n_dq;    // (workgroups of 64 rows)
    const bool causal = mode == NNTILE_HIP_MASK_CAUSAL;
    if(!causal && mode != NNTILE_HIP_MASK_NONE)
    {
        return apart <= 2 * kBwdCUs ? BWD_HALVED_APART
            : head == 64 && both <= 2 * kBwdCUs ? BWD_HALVED_BOTH : BWD_WHOLE_STEPS;
    }
    // (the first of those lines: short walks of entries that do not come in eights)
    if(apart > 2 * kBwdCUs && entries % 8 != 0 && bwd_longest_walk(p) <= 16)
    {
        return BWD_WHOLE_STEPS;
    }
    if(head == 64)
    {
        const bool few = both <= (causal ? 4 : 2) * kBwdCUs
            || (p.kv_group >= (causal ? 2 : 4) && n_dkv <= (causal ? 256 : 208));
        return apart <= kBwdCUs ? BWD_HALVED_APART : few ? BWD_HALVED_BOTH : BWD_WHOLE_STEPS;
    }
    // (the second: rectangular calls of short walks)
    if(p.q_seq != p.k_seq && bwd_longest_walk(p) < kBwdLongWalk)
    {
        return BWD_WHOLE_STEPS;
    }
    const bool few = apart <= (causal ? 3 : 2) * kBwdCUs
        || (p.kv_group >= 4 && n_dkv <= (causal ? 256 : 128));
    return few ? BWD_HALVED_APART : BWD_WHOLE_STEPS;
}

// Workgroups of two groups of wavefronts (sdpa_bwd_kernel, GROUPS == 2), where one
// computes dK and dV: the workgroups that own keys walk
// every query of a group's heads, under a causal mask those of the first keys all of
// them, and a launch that has not enough of them to fill the chip ends with their walks.
// One group (and operands not read ahead) / two, us, bf16, one box: head 128, causal, 64
// query heads on 16, 800 rows 150 / 91, 2 500 503 / 457, two groups of eight, 4 096 rows,
// 1 268 / 728; 32 heads, 800 rows 50 / 42, 8 heads, 4 096 rows 190 / 134; head 64 70 / 54,
// 235 / 225, 546 / 405, 26.5 / 26.4, 95 / 77.  Without a mask every walk is as long:
// grouped 800 rows 154 / 98 (head 64 72 / 59), two groups of eight, 4 096 rows, 1 305 / 787
// (550 / 415), but one head a group 800 rows 53 / 57 (28 / 34), and from 208 workgroups of
// head 64 on 161 / 167.
static bool bwd_two_groups_fused(int64_t n_dkv, const BwdParams &p, int mode)
{
    const bool few = mode == NNTILE_HIP_MASK_CAUSAL ? n_dkv <= kBwdCUs
        : p.kv_group > 1 && n_dkv <= kBwdCUs * 3 / 4;
    return few && bwd_longest_walk(p) >= kBwdLongWalk;
}

// The same from the workgroups of 128 rows, which become those of 64 where it is halved.
static int bwd_halved(const BwdParams &p, int head, int mode, int64_t &n_dkv, int64_t &n_dq)
{
    constexpr int kHalf = kDkvRows / 2;
    const int64_t entries = n_dkv / ((p.k_seq + kDkvRows - 1) / kDkvRows);
    const int64_t n_dkv64 = entries * ((p.k_seq + kHalf - 1) / kHalf);
    const int64_t n_dq64 = n_dq / ((p.q_seq + kDkvRows - 1) / kDkvRows) * ((p.q_seq + kHalf - 1) / kHalf);
    const int how = bwd_halved(p, head, mode, entries, n_dkv64, n_dq64);
    if(how != BWD_WHOLE_STEPS)
    {
        n_dkv = n_dkv64;
        n_dq = n_dq64;
    }
    return how;
}

template<typename Kernel, typename Params>
static int launch_bwd_wgs(hipStream_t stream, Kernel kernel, const Params &p, int64_t n_wgs, int groups,
        int64_t n_dkv, int64_t n_dq)
{
    hipLaunchKernelGGL(kernel, dim3((unsigned)n_wgs), dim3(groups * kDkvThreads), 0, stream, p,
            (unsigned)n_dkv, (unsigned)n_dq);
    return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
}

// Whether a gradient lies in the memory of A.  The launch in front is done with A before
// the first gradient is written, so such calls are right with it, and only with it.
static bool bwd_writes_into_A(const BwdParams &p, int head)
{
    const int64_t q_bytes = (int64_t)p.batch * p.q_seq * head * 2;
    const int64_t k_bytes = (int64_t)(p.batch / p.kv_group) * p.k_seq * head * 2;
    const uintptr_t a = reinterpret_cast<uintptr_t>(p.A);
    auto meets = [&](const void *out, int64_t bytes)
    {
        const uintptr_t o = reinterpret_cast<uintptr_t>(out);
        return o < a + (uintptr_t)q_bytes && a < o + (uintptr_t)bytes;
    };
    return meets(p.dQ, q_bytes) || meets(p.dK, k_bytes) || meets(p.dV, k_bytes);
}

// The form without the launch in front, where steps are halved and no workgroup needs more
// than kBwdOwnRows (measured there); false: the call is for the other forms.
template<typename T, int HEAD, int MODE>
static bool launch_bwd_short(hipStream_t stream, const BwdParams &p, int64_t n_dkv, int64_t n_dq, int &rc)
{
    if constexpr(HEAD >= 64)
    {
        if(p.q_seq > kBwdOwnRows / p.kv_group || p.k_seq > kBwdOwnRows || bwd_writes_into_A(p, HEAD))
        {
            return false;
        }
        const int how = bwd_halved(p, HEAD, MODE, n_dkv, n_dq);
        if(how == BWD_HALVED_APART)
        {
            rc = launch_bwd_wgs(stream, sdpa_bwd_kernel<T, HEAD, MODE, false, false, 1, 2, true>, p,
                    2 * n_dkv + n_dq, 1, n_dkv, n_dq);
            return true;
        }
        if constexpr(HEAD == 64)
        {
            if(how == BWD_HALVED_BOTH)
            {
                rc = launch_bwd_wgs(stream, sdpa_bwd_kernel<T, HEAD, MODE, false, true, 1, 2, true>, p,
                        n_dkv + n_dq, 1, n_dkv, n_dq);
                return true;
            }
        }
    }
    return false;
}

// The gradient launch, the same for one allocation (GRID false) and for tiles.
template<typename T, int HEAD, int MODE, bool GRID>
static int launch_bwd_kernel(hipStream_t stream,
        const std::conditional_t<GRID, BwdGridParams, BwdParams> &p, int64_t n_dkv, int64_t n_dq)
{
    constexpr bool ANALYTIC = MODE == NNTILE_HIP_MASK_NONE || MODE == NNTILE_HIP_MASK_CAUSAL;
    auto launch = [&](auto kernel, int64_t n_wgs, int groups) -> int
    {
        return launch_bwd_wgs(stream, kernel, p, n_wgs, groups, n_dkv, n_dq);
    };
    if constexpr(HEAD >= 64)
    {
        const int how = bwd_halved(p, HEAD, MODE, n_dkv, n_dq);
        if(how == BWD_HALVED_APART)
        {
            return launch(sdpa_bwd_kernel<T, HEAD, MODE, GRID, false, 1, 2>, 2 * n_dkv + n_dq, 1);
        }
        if constexpr(HEAD == 64)
        {
            if(how == BWD_HALVED_BOTH)
            {
                return launch(sdpa_bwd_kernel<T, HEAD, MODE, GRID, true, 1, 2>, n_dkv + n_dq, 1);
            }
        }
    }
    if constexpr(kBwdFusedKeys<HEAD, MODE>)
    {
        // One set of key-owning workgroups for both gradients (seven products
        // instead of eight) once the three sets would not all be resident at
        // the same time; below that the longest workgroup sets the time, and
        // the separate sets have the shorter ones.
        if(2 * n_dkv + n_dq > 2 * kBwdCUs)
        {
            if constexpr(HEAD >= 64 && ANALYTIC)
            {
                if(bwd_two_groups_fused(n_dkv, p, MODE))
                {
                    return launch(sdpa_bwd_kernel<T, HEAD, MODE, GRID, true, 2>, n_dkv + n_dq, 2);
                }
            }
            return launch(sdpa_bwd_kernel<T, HEAD, MODE, GRID, true>, n_dkv + n_dq, 1);
        }
    }
    return launch(sdpa_bwd_kernel<T, HEAD, MODE, GRID>, 2 * n_dkv + n_dq, 1);
}

template<typename T, int HEAD, int MODE>
static int launch_bwd_mode(hipStream_t stream, const BwdParams &p)
{
    const int64_t q_blocks = (p.q_seq + kBwdRows - 1) / kBwdRows;
    const int64_t k_blocks = (p.k_seq + kDkvRows - 1) / kDkvRows;
    const int64_t kv_batch = p.batch / p.kv_group;
    const int64_t n_dq = (int64_t)p.batch * q_blocks, n_dkv = kv_batch * k_blocks;
    if(n_dq <= 0 || n_dkv <= 0 || n_dq > 0x3fffffff || n_dkv > 0x3fffffff
            || (int64_t)p.batch * p.q_seq * (HEAD / 8) / 256 > 0x7ffffffe)
    {
        return NNTILE_HIP_EINVAL;
    }
    int rc;
    if(launch_bwd_short<T, HEAD, MODE>(stream, p, n_dkv, n_dq, rc))
    {
        return rc;
    }
    BwdPreludeParams pre = prelude_params(p, p.q_seq, 1);
    pre.dA[0] = p.dA;
    pre.A[0] = p.A;
    if((MODE == NNTILE_HIP_MASK_ADDITIVE || MODE == NNTILE_HIP_MASK_BOOL)
            && p.mask_class != nullptr)
    {
        pre.table = const_cast<uint8_t *>(p.mask_class);
        pre.class_ld = p.class_ld;
        const int64_t n_cls = ((p.q_seq + kBwdStep - 1) / kBwdStep) * p.class_ld;
        if(n_cls > 0x3fffffff)
        {
            return NNTILE_HIP_EINVAL;
        }
        pre.n_class_wgs = (int32_t)n_cls;
    }
    rc = launch_prelude<T, HEAD, MODE>(stream, pre, 1);
    if(rc != NNTILE_HIP_OK)
    {
        return rc;
    }
    return launch_bwd_kernel<T, HEAD, MODE, false>(stream, p, n_dkv, n_dq);
}

// The grid form: the row dots tile by tile (each tile's A and dA are one
// allocation, and D follows the layout of lse), then the one gradient launch.
template<typename T, int HEAD, int MODE>
static int launch_bwd_grid_mode(hipStream_t stream, const BwdGridParams &p,
        const void *const *A_tiles, int n_q_tiles)
{
    const int64_t q_blocks = (p.q_seq + kBwdRows - 1) / kBwdRows;
    const int64_t k_blocks = (p.k_seq + kDkvRows - 1) / kDkvRows;
    const int64_t kv_batch = p.batch / p.kv_group * p.n_slabs;
    const int64_t n_dq = (int64_t)p.batch * p.n_slabs * q_blocks, n_dkv = kv_batch * k_blocks;
    if(n_dq <= 0 || n_dkv <= 0 || n_dq > 0x3fffffff || n_dkv > 0x3fffffff
            || (int64_t)p.batch * p.q_tile * (HEAD / 8) / 256 > 0x7ffffffe)
    {
        return NNTILE_HIP_EINVAL;
    }
    if(p.n_slabs == 1 && n_q_tiles == 1 && p.n_kv_tiles == 1)
    {
        // (one tile an axis is one allocation)
        BwdParams one = p;
        one.Q = p.Qt[0];
        one.K = p.Kt[0];
        one.V = p.Vt[0];
        one.A = A_tiles[0];
        one.dA = p.dAt[0];
        one.lse = p.lset[0];
        one.dQ = p.dQt[0];
        one.dK = p.dKt[0];
        one.dV = p.dVt[0];
        int rc;
        if(launch_bwd_short<T, HEAD, MODE>(stream, one, n_dkv, n_dq, rc))
        {
            return rc;
        }
    }
    BwdPreludeParams pre = prelude_params(p, p.q_tile, n_q_tiles);
    for(int t = 0; t < p.n_slabs * n_q_tiles; ++t)
    {
        pre.dA[t] = p.dAt[t];
        pre.A[t] = A_tiles[t];
    }
    const int pre_rc = launch_prelude<T, HEAD, MODE>(stream, pre, p.n_slabs * n_q_tiles);
    if(pre_rc != NNTILE_HIP_OK)
    {
        return pre_rc;
    }
    return launch_bwd_kernel<T, HEAD, MODE, true>(stream, p, n_dkv, n_dq);
}

template<typename T, int HEAD>
static int launch_bwd_grid_head(hipStream_t stream, const BwdGridParams &p,
        const void *const *A_tiles, int n_q_tiles, int mode)
{
    switch(mode)
    {
        case NNTILE_HIP_MASK_NONE:
            return launch_bwd_grid_mode<T, HEAD, NNTILE_HIP_MASK_NONE>(stream, p, A_tiles,
                    n_q_tiles);
        case NNTILE_HIP_MASK_CAUSAL:
            return launch_bwd_grid_mode<T, HEAD, NNTILE_HIP_MASK_CAUSAL>(stream, p, A_tiles,
                    n_q_tiles);
        default:
            return NNTILE_HIP_EINVAL;
    }
}

// The caller has checked: every tile but the last of an axis holds q_tile /
// k_tile rows, both multiples of 128 unless the axis is one tile.
template<typename T>
int launch_bwd_grid_16bit(hipStream_t stream, const BwdGridParams &p,
        const void *const *A_tiles, int n_q_tiles, int head, int mode)
{
    switch(head)
    {
        case 32:
            return launch_bwd_grid_head<T, 32>(stream, p, A_tiles, n_q_tiles, mode);
        case 64:
            return launch_bwd_grid_head<T, 64>(stream, p, A_tiles, n_q_tiles, mode);
        case 128:
            return launch_bwd_grid_head<T, 128>(stream, p, A_tiles, n_q_tiles, mode);
        default:
            return NNTILE_HIP_EUNSUPPORTED;
    }
}

template int launch_bwd_grid_16bit<Bf16>(hipStream_t, const BwdGridParams &, const void *const *,
        int, int, int);
template int launch_bwd_grid_16bit<Fp16>(hipStream_t, const BwdGridParams &, const void *const *,
        int, int, int);

template<typename T, int HEAD>
static int launch_bwd_head(hipStream_t stream, const BwdParams &p, int mode)
{
    switch(mode)
    {
        case NNTILE_HIP_MASK_ADDITIVE:
            return launch_bwd_mode<T, HEAD, NNTILE_HIP_MASK_ADDITIVE>(stream, p);
        case NNTILE_HIP_MASK_NONE:
            return launch_bwd_mode<T, HEAD, NNTILE_HIP_MASK_NONE>(stream, p);
        case NNTILE_HIP_MASK_CAUSAL:
            return launch_bwd_mode<T, HEAD, NNTILE_HIP_MASK_CAUSAL>(stream, p);
        case NNTILE_HIP_MASK_BOOL:
            return launch_bwd_mode<T, HEAD, NNTILE_HIP_MASK_BOOL>(stream, p);
        default:
            return NNTILE_HIP_EINVAL;
    }
}

template<typename T>
int launch_bwd_16bit(hipStream_t stream, const BwdParams &p, int head, int mode)
{
    switch(head)
    {
        case 32:
            return launch_bwd_head<T, 32>(stream, p, mode);
        case 64:
            return launch_bwd_head<T, 64>(stream, p, mode);
        case 128:
            return launch_bwd_head<T, 128>(stream, p, mode);
        default:
            return NNTILE_HIP_EUNSUPPORTED;
    }
}

template int launch_bwd_16bit<Bf16>(hipStream_t, const BwdParams &, int, int);
template int launch_bwd_16bit<Fp16>(hipStream_t, const BwdParams &, int, int);

} // namespace nntile_hip
