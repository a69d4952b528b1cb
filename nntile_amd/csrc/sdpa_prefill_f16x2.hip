// Prefill attention forward for fp32 tiles on the fp16 matrix units of gfx950.
//
// The fp32 matrix instructions run at 157 TFLOP/s, the fp16 ones at 2500.  A
// float is, to 22 bits, the sum of two fp16 values: x = h + l with h = fp16(x),
// l = fp16(x - h), what is left is at most 2^-23 of x.  Of the four products of
// two such sums l.h, h.l and h.h are added up in fp32 by the matrix unit; l.l is
// at most 2^-22 of the product, 2^-25 in the mean.  Three fp16 products cost
// 3/16 of an fp32 one, so the ceiling moves from 157 to 833 TFLOP/s, and a sum
// of head (or key) products is rounded a fifth as often.  (The method: Markidis
// et al., "NVIDIA Tensor Core Programmability, Performance & Precision", 2018;
// Ootomo and Yokota, "Recovering single precision accuracy from Tensor Cores
// while surpassing the FP32 theoretical peak performance", 2022.)
//
// fp16 holds 22 bits of x in two values for 2^-3 <= |x| < 2^16, and 2^-25
// absolutely below, so the values are moved there by powers of two, which are
// exact: a row of Q so that its largest value is in [2^13, 2^14), K and V so that
// the largest of a workgroup's first step is in [2^11, 2^12), the probabilities
// (at most 1) by 2^15.  A workgroup takes its keys with fp32 matrix instructions
// where that does not do.  From the start: rows whose scores the pieces may not carry
// (below), Q, K or V beyond 2^40, V below 2^-40.  A second time, found on the way or in
// the results: infinities and NaN, later keys or values more than 16 times larger
// than those of the first step (an overflow makes them NaN), eight values of a channel
// of V that are split together all 2^-13 times the first step's largest or less, rows
// of the output that are as small.  What stays is 2^-22 of a product and, absolutely,
// 2^-23 of a score (below) and 2^-23 of a probability times the largest of the eight
// values that are split together.
//
// Scores: what a piece loses absolutely, 2^-25 of a scaled value, counts by what it
// is multiplied with.  With q and k the largest values of a row of Q and of the first
// keys that is up to q k 2^-37 in a score (rounding errors of random signs in every
// channel), and where large channels of one meet small ones of the other the score
// may be that and little else.  So rows with q k above 2^12 to 2^14 (the powers of
// two say which, in front of the walk) go to fp32 from the start; below, the errors
// of a score stay under 2^-23, or 2^-21 where all later keys are 16 times larger.
//
// S^T = K Q^T and O^T += V^T P^T with a lane owning one query, as in the other
// prefill kernels.  A workgroup holds QW blocks of 32 queries; a key step is G
// blocks of 32 keys, and wavefront (q, g) takes query block q against key block
// g.  K and V are split once per workgroup on their way into LDS, where each
// piece lies in the order in which a matrix operand is read (1 KB a fragment,
// 16 bytes a lane: no bank conflicts, V transposed on the way in), Q once into
// registers, the probabilities where they are.  A pass of the loop computes the
// scores of step i+1 and the output of step i on the matrix unit; in slices
// behind its instructions run the softmax of step i and the splitting of
// K(i+2) and V(i+1), whose rows were requested into registers a pass before.
// Two LDS buffers each for K and V: one barrier a pass.
//
// What bounds it: the vector port.  A matrix instruction takes it for 16 clocks
// and every vector instruction for 4; a pass at head 64 is 24 of the first and
// about 175 (8 x 1: 120) of the second for 32 x 32 scores, 1 090 clocks against 768
// of the matrix unit; two wavefronts a SIMD come to 70 % of that.  (Three bf16
// pieces, which need no powers of two: twice the products and 11 instead of 6
// vector instructions for a pair of values, 50 us where this took 41 at 48 x 1024
// x 64.)
#include <cmath>
#include <type_traits>

#include "sdpa_mask_scan.hpp"

namespace nntile_hip
{

constexpr int kX2Rows = 32;         // queries of a wavefront, keys of a wavefront's step
// Probabilities are scaled by 2^4 in the exponential - the arguments that matter lie
// within 4 of zero, where a float is finest (2^14: errors of A a fifth larger than with
// fp32 products, of lse 5 %) - and by 2^11 more as they are split: what their pieces
// lose is below 2^-40.  (With 2^4 alone it was 2^-29, and rows that a first key with
// little of a value takes most of were made of those errors: 13 above the others'
// scores, 700 keys: 2.2e-5 where fp32 products have 4.0e-7.)
constexpr int kX2PExp = 4;
constexpr float kX2PPieces = 0x1p11f;
// The inverse of the product of a row's power of two and that of K up to which their
// scores are taken from pieces: largest values of 2^12 to 2^14 as a product.
constexpr float kX2Scores = 0x1p-12f;

// The two fp16 pieces of eight floats times a power of two, as matrix operands.
struct Split8
{
    u32x4 h, l;
    // (fma with an fp16 operand: no conversion back.  Fmas with an fp16 result, four
    // instructions instead of six, take 6 to 10 % longer in all.)
    __device__ __forceinline__ void pair(int i, float a, float b, float scale)
    {
        h[i] = Fp16::pack2(a * scale, b * scale);
        l[i] = Fp16::pack2(fmaf(a, scale, -lo_half(h[i])), fmaf(b, scale, -hi_half(h[i])));
    }
    static __device__ __forceinline__ float lo_half(uint32_t v)
    {
        return Fp16::to_float((uint16_t)(v & 0xffffu));
    }
    static __device__ __forceinline__ float hi_half(uint32_t v)
    {
        return Fp16::to_float((uint16_t)(v >> 16));
    }
};

// acc += a.b; one of the three products, the smallest first
__device__ __forceinline__ f32x16 product(int n, const Split8 &a, const Split8 &b, f32x16 acc)
{
    const u32x4 x = n == 0 ? a.l : a.h, y = n == 1 ? b.l : b.h;
    return Fp16::mfma(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), acc);
}

// The power of two that moves `largest` into [2^(to-1), 2^to) and its inverse;
// false when it is out of the range that is moved (then 1).  LEAST: what is below
// 2^-40, zeros among them, is moved as if it were that (the factors of a score:
// times one below 2^40, what the pieces then lose is below 2^-30).
template<bool LEAST>
__device__ __forceinline__ bool power_to(float largest, int to, float &scale, float &inverse)
{
    scale = inverse = 1.0f;
    if(LEAST)
    {
        largest = fmaxf(largest, 0x1p-40f);
    }
    if(!(largest >= 0x1p-40f && largest < 0x1p40f))
    {
        return false;
    }
    const int e = __builtin_amdgcn_frexp_expf(largest);     // largest in [2^(e-1), 2^e)
    scale = __uint_as_float((uint32_t)(127 + to - e) << 23);
    inverse = __uint_as_float((uint32_t)(127 - to + e) << 23);
    return true;
}

// PARTS: the workgroup takes one of p.n_parts ranges of the keys and leaves its
// triple in memory (PrefillParams::part_o) for launch_parts_merge.
template<int HEAD, int MODE, int QW, int G, bool PARTS = false>
__global__ __launch_bounds__(64 * QW * G, HEAD == 128 && QW == 2 ? 1 : 2)
void sdpa_prefill_f16x2_kernel(const PrefillParams p)
{
    constexpr int THREADS = 64 * QW * G;
    constexpr int QROWS = kX2Rows * QW;     // queries per workgroup
    constexpr int KEYS = kX2Rows * G;       // keys per step of the workgroup
    constexpr int CH = HEAD / 16;           // matrix instructions along the head (scores)
    constexpr int DB = HEAD / 32;           // blocks of the head (output)
    constexpr int HG = HEAD / 8;            // groups of 8 head values
    constexpr int GB = 2 * kX2Rows * HEAD * 2;      // bytes of a key block's pieces
    // pieces of 8 values that a thread splits per step of K, and of V
    constexpr int UNITS = KEYS * HG;
    constexpr int UPT = (UNITS + THREADS - 1) / THREADS;
    constexpr int NS = 3 * CH, NP = 6 * DB;         // matrix instructions of scores and output
    // Rows are requested into SETS sets of registers in turn, SETS passes before they
    // are split (what a lane holds at head 128 leaves room for one).
    constexpr int AHEAD_FR = HEAD == 64 ? 2 : 1;
    constexpr int SETS = HEAD >= 128 ? 1 : 2;
    constexpr bool EXPLICIT = (MODE == NNTILE_HIP_MASK_ADDITIVE
            || MODE == NNTILE_HIP_MASK_BOOL);
    static_assert(!PARTS || !EXPLICIT, "parts: analytic masks");

    constexpr int BUF = G * GB;             // K(0) K(1) V(0) V(1)
    __shared__ __attribute__((aligned(1024))) char lds[4 * BUF];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31;
    const int half = lane >> 5;
    const int qw = wave % QW, grp = wave / QW;

    const int q_blocks = p.n_q_tiles * p.q_blocks_per_tile;
    const int batch_all = p.batch * p.n_slabs;
    int wg = blockIdx.x;
    int part = 0;
    if constexpr(PARTS)
    {
        const int per_part = (int)gridDim.x / p.n_parts;
        part = wg / per_part;
        wg -= part * per_part;
    }
    const int64_t part_k0 = PARTS ? (int64_t)part * p.part_keys : 0;
    const int64_t k_seq = PARTS ? min((int64_t)p.part_keys, p.k_seq - part_k0) : p.k_seq;
    const int64_t k_tile = PARTS ? k_seq : p.k_tile;
    const int64_t k_pos0 = p.k_pos0 + part_k0;
    const bool overwrite = PARTS || p.overwrite;
    // Longest query blocks first, all batch entries of a block before the next
    // block: CUs that become free take what is left in the order of its length,
    // and a number of entries that is a multiple of 8 keeps an entry on one XCD.
    int b = wg % batch_all;
    const int qblk = q_blocks - 1 - wg / batch_all;
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
    const int64_t q_len = min(p.q_tile, p.q_seq - (int64_t)qt * p.q_tile);
    const int64_t q_row0 = (int64_t)qb * QROWS;
    if(q_row0 >= q_len)
    {
        return;
    }
    const int kvb = kv_entry(b, p.n_batch, p.kv_group);
    const float *Qt = static_cast<const float *>(p.Q[q_tile0 + qt]) + (int64_t)b * q_len * HEAD;
    const int64_t wave_q = q_row0 + qw * kX2Rows;
    const bool q_ok = wave_q + col < q_len;
    // this lane's query row (the tile's first for a lane that has none)
    auto my_row = [&]() __attribute__((always_inline)) -> int64_t
    {
        return q_ok ? wave_q + col : 0;
    };

    // ---- the steps to walk -----------------------------------------------------
    const int64_t last_k_len = k_seq - (int64_t)(p.n_kv_tiles - 1) * k_tile;
    int n_steps = (p.n_kv_tiles - 1) * p.k_blocks_per_tile
        + (int)((last_k_len + KEYS - 1) / KEYS);
    const int64_t wg_qpos_hi = p.q_pos0 + (int64_t)qt * p.q_tile + min(q_row0 + QROWS, q_len) - 1;
    const int64_t wave_qpos_lo = p.q_pos0 + (int64_t)qt * p.q_tile + wave_q;
    if(MODE == NNTILE_HIP_MASK_CAUSAL)
    {
        const int64_t hi = wg_qpos_hi + p.causal_offset - k_pos0;
        if(hi < 0)
        {
            if(!overwrite)
            {
                return;
            }
            n_steps = 0;    // nothing visible: the epilogue writes empty rows
        }
        const int64_t kt_hi = hi < 0 ? (int64_t)p.n_kv_tiles : hi / k_tile;
        if(kt_hi < p.n_kv_tiles)
        {
            const int64_t in_tile = hi - kt_hi * k_tile;
            n_steps = min(n_steps, (int)(kt_hi * p.k_blocks_per_tile + in_tile / KEYS + 1));
        }
    }
    // A mask given as values: the workgroup's rows of it are looked over once;
    // hidden steps at either end are not walked, open ones read no mask values.
    int n_skip = 0;
    unsigned long long not_open = ~0ull;
    if constexpr(EXPLICIT)
    {
        constexpr int ES = (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 4 : 1;
        if(n_steps > 0 && k_seq * ES >= 16 && p.mask_ld * ES * QROWS < (int64_t)(1 << 30))
        {
            __shared__ unsigned long long scan_words[2 * THREADS / 64];
            unsigned long long not_hidden;
            mask_scan_steps<ES, THREADS / 64, KEYS>(static_cast<const char *>(p.mask)
                    + q_row0 * p.mask_ld * ES, (uint32_t)(p.mask_ld * ES),
                    (int)min((int64_t)QROWS, q_len - q_row0), (int)k_seq * ES, 0, n_steps,
                    (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 0u : 0x01010101u,
                    (MODE == NNTILE_HIP_MASK_ADDITIVE) ? 0xff800000u : 0u, scan_words, not_open,
                    not_hidden);
            if(not_hidden == 0ull)
            {
                if(!overwrite)
                {
                    return;
                }
                n_steps = 0;        // the epilogue writes empty rows
            }
            else
            {
                if((not_hidden >> 63) == 0ull)
                {
                    n_steps = min(n_steps, 64 - __builtin_clzll(not_hidden));
                }
                n_skip = min(__builtin_ctzll(not_hidden), n_steps - 1);
                n_steps -= n_skip;
            }
        }
    }

    // ---- where the rows of a step come from -------------------------------------
    struct StepSource
    {
        const float *K, *V;     // first row of the step
        int step, kt, rows_left;        // rows of the tile kt from this step on
        int64_t k_row0, k_pos;  // the step's first key: in its tile, on the key axis
    };
    auto tile_of = [&](StepSource &src) __attribute__((always_inline))
    {
        const int64_t k_len = min(k_tile, k_seq - (int64_t)src.kt * k_tile);
        const int64_t entry_rows = p.kv_rows > 0 ? p.kv_rows : k_len;   // (a cache is one tile)
        const int64_t off = ((int64_t)kvb * entry_rows + part_k0 + src.k_row0) * HEAD;
        src.K = static_cast<const float *>(p.K[k_tile0 + src.kt]) + off;
        src.V = static_cast<const float *>(p.V[k_tile0 + src.kt]) + off;
        src.rows_left = (int)(k_len - src.k_row0);
        src.k_pos = k_pos0 + (int64_t)src.kt * k_tile + src.k_row0;
    };
    // (one division, in front of the walk; then from step to step)
    auto first_step = [&]() __attribute__((always_inline)) -> StepSource
    {
        StepSource src;
        src.step = 0;
        src.kt = p.n_kv_tiles == 1 ? 0 : n_skip / p.k_blocks_per_tile;
        src.k_row0 = (int64_t)(n_skip - src.kt * p.k_blocks_per_tile) * KEYS;
        tile_of(src);
        return src;
    };
    // (steps past the last are that one again: what is read there nobody uses)
    auto advance = [&](StepSource &src) __attribute__((always_inline))
    {
        if(src.step + 1 < n_steps)
        {
            ++src.step;
            src.K += KEYS * HEAD;
            src.V += KEYS * HEAD;
            src.rows_left -= KEYS;
            src.k_row0 += KEYS;
            src.k_pos += KEYS;
            if(src.rows_left <= 0)
            {
                ++src.kt;
                src.k_row0 = 0;
                tile_of(src);
            }
        }
    };

    // ---- global memory -> registers -> pieces in LDS ------------------------------
    // K unit u: key u / HG of the step, head values 8 * (u % HG) .. +7.  Its two
    // pieces go to fragment (head group / 2) of the key's block; inside the 512
    // bytes of a lane half the keys' places are permuted so that the 16 lanes of a
    // write hit 16 different ones, and so do those of a read.
    // V unit u: head value u % HEAD, keys of slot group u / HEAD - the eight keys
    // that a lane half's score registers hold of 16 (4 * half .. +3 and 8 further).
    // Rows past the end of the tile are its last row (V: zeros, where all eight are past
    // it): their scores are masked, so their probabilities are exactly 0.
    constexpr int KSW = 16 / HG;            // keys of a row of 16 lanes
    auto k_place = [](int key, int hg) __attribute__((always_inline)) -> int
    {
        return key ^ hg ^ ((key & (KSW - 1)) * (HG % 16));
    };
    // Units i * THREADS + tid of a thread: a power of two of keys (of slot groups)
    // apart, so what follows from i is an offset known when this is compiled.
    constexpr int KSTRIDE = THREADS / HG, SSTRIDE = THREADS / HEAD;
    static_assert(UPT == 1 || (KSTRIDE >= 16 && SSTRIDE >= 1), "units of a thread");
    auto k_lds = [](int i) { return i * KSTRIDE / 32 * GB + i * KSTRIDE % 32 * 16; };
    auto v_lds = [](int i)
    {
        const int slots = i * SSTRIDE;
        return (slots >> 2) * GB + ((slots >> 1) & 1) * DB * 1024 + (slots & 1) * 512;
    };
    auto v_rows = [](int slots) { return (slots >> 1) * 16 + (slots & 1) * 4; };
    StepSource k_src = {}, v_src = {}, s_src = {};      // the rows requested last, the scores
    f32x4 k_raw[SETS][UPT][2];
    float v_raw[SETS][UPT][8];
    float k_scale = 1.0f, v_scale = 1.0f, v_back = 1.0f;
    uint32_t k_goff, v_goff;
    int k_at, v_at;
    {
        const int u = min(tid, UNITS - 1);
        const int key = u / HG, hg = u % HG, d = u % HEAD, slots = u / HEAD;
        k_goff = (uint32_t)(key * HEAD + hg * 8) * 4;
        k_at = (key / kX2Rows) * GB + (hg / 2) * 1024 + (hg % 2) * 512
            + k_place(key % kX2Rows, hg) * 16;
        v_goff = (uint32_t)(v_rows(slots) * HEAD + d) * 4;
        v_at = (slots >> 2) * GB + (((slots >> 1) & 1) * DB + d / 32) * 1024
            + ((slots & 1) * 32 + d % 32) * 16;
    }
    // One load instruction of a step's rows: n of the 2 * UPT (K), of the 8 * UPT (V).
    // (32-bit offsets on a base common to the wavefront.  The last rows of a tile go
    // in one piece, load_k_tail / load_v_tail.)
    auto load_k_piece = [&](int set, int n) __attribute__((always_inline))
    {
        const char *at = reinterpret_cast<const char *>(k_src.K) + n / 2 * KSTRIDE * HEAD * 4 + n % 2 * 16;
        k_raw[set][n / 2][n % 2] = *reinterpret_cast<const f32x4 *>(at + k_goff);
    };
    auto load_v_piece = [&](int set, int n) __attribute__((always_inline))
    {
        const int e = n % 8;
        const char *at = reinterpret_cast<const char *>(v_src.V)
            + (v_rows(n / 8 * SSTRIDE) + (e < 4 ? e : e + 4)) * HEAD * 4;
        v_raw[set][n / 8][e] = *reinterpret_cast<const float *>(at + v_goff);
    };
    auto load_k_tail = [&](int set) __attribute__((always_inline))
    {
        uint32_t goff = k_goff;
        asm volatile("" : "+v"(goff));      // (worked out here, not kept in registers or
                                            // scratch memory through the walk)
#pragma unroll
        for(int i = 0; i < UPT; ++i)
        {
            const int key = (int)(goff / (HEAD * 4)) + i * KSTRIDE;
            const uint32_t off = goff + (uint32_t)(i * KSTRIDE * HEAD * 4)
                - (uint32_t)(max(key - (k_src.rows_left - 1), 0) * HEAD * 4);
            const char *at = reinterpret_cast<const char *>(k_src.K) + off;
            k_raw[set][i][0] = *reinterpret_cast<const f32x4 *>(at);
            k_raw[set][i][1] = *reinterpret_cast<const f32x4 *>(at + 16);
            // (waits, and keeps the compiler from making one set of loads with
            // 64-bit addresses out of the two forms)
            asm volatile("" : "+v"(k_raw[set][i][0]), "+v"(k_raw[set][i][1]));
        }
    };
    // Units of the last one or two rows of a tile do not say how small a channel is: one
    // value in 4000 of N(0, 1) is below what look_at_unit asks for, so one in 15 heads
    // of 128 would walk its keys again for one of them (24 heads, 710 x 1781, head 128, 78 us
    // or 330).  They hold that much in rows past the end, unless their values are below
    // 2^-12 or nothing else speaks for the channel (a first step of one or two rows).
    constexpr float LEAST = 0x1p-2f;
    auto few_rows = [&](int set, uint32_t goff) __attribute__((always_inline))
    {
#pragma unroll
        for(int i = 0; i < UPT; ++i)
        {
            const int rows = v_src.rows_left - (int)(goff / (HEAD * 4)) - v_rows(i * SSTRIDE);
            const float largest = fmaxf(__builtin_fabsf(v_raw[set][i][0]), __builtin_fabsf(v_raw[set][i][1]));
            const bool alone = v_src.step == 0 && v_src.rows_left <= 2;
            if(rows <= 2 && !alone && largest >= 0x1p-10f * LEAST * v_back)
            {
                v_raw[set][i][7] = LEAST * v_back;
            }
        }
    };
    auto load_v_tail = [&](int set) __attribute__((always_inline))
    {
        uint32_t goff = v_goff;
        asm volatile("" : "+v"(goff));      // (as above)
#pragma unroll
        for(int i = 0; i < UPT; ++i)
        {
#pragma unroll
            for(int e = 0; e < 8; ++e)
            {
                const int add = v_rows(i * SSTRIDE) + (e < 4 ? e : e + 4);
                const int key = (int)(goff / (HEAD * 4)) + add;
                const uint32_t off = goff + (uint32_t)(add * HEAD * 4)
                    - (uint32_t)(max(key - (v_src.rows_left - 1), 0) * HEAD * 4);
                v_raw[set][i][e] = *reinterpret_cast<const float *>(
                        reinterpret_cast<const char *>(v_src.V) + off);
            }
#pragma unroll
            for(int e = 0; e < 8; ++e)
            {
                asm volatile("" : "+v"(v_raw[set][i][e]));      // (as above)
            }
            if((int)(goff / (HEAD * 4)) + v_rows(i * SSTRIDE) >= v_src.rows_left)
            {
#pragma unroll
                for(int e = 0; e < 8; ++e)
                {
                    v_raw[set][i][e] = 0.0f;
                }
            }
        }
        if(v_src.step > 0)      // (the first step: once its power of two is known)
        {
            few_rows(set, goff);
        }
    };
    auto load_k = [&](int set) __attribute__((always_inline))
    {
        if(k_src.rows_left >= KEYS)
        {
#pragma unroll
            for(int n = 0; n < 2 * UPT; ++n)
            {
                load_k_piece(set, n);
            }
        }
        else
        {
            load_k_tail(set);
        }
    };
    auto load_v = [&](int set) __attribute__((always_inline))
    {
        if(v_src.rows_left >= KEYS)
        {
#pragma unroll
            for(int n = 0; n < 8 * UPT; ++n)
            {
                load_v_piece(set, n);
            }
        }
        else
        {
            load_v_tail(set);
        }
    };

    // ---- this lane's operands and the powers of two --------------------------------
    Split8 qf[CH];
    float qk_back = 1.0f;       // scores / (what the matrix unit computes)
    bool odd = false;           // something that the pieces cannot carry
    __shared__ int any_odd, any_large;
    if(n_steps > 0)
    {
        k_src = v_src = s_src = first_step();
        __shared__ float first_max[2 * THREADS / 64];
        if(tid == 0)
        {
            any_odd = any_large = 0;
        }
        load_k(0);
        load_v(0);
        const float *Qrow = Qt + my_row() * HEAD;
        f32x4 raw[2 * CH];
        float q_max = 0.0f;
#pragma unroll
        for(int j = 0; j < 2 * CH; ++j)
        {
            raw[j] = *reinterpret_cast<const f32x4 *>(Qrow + 16 * (j / 2) + 8 * half + 4 * (j % 2));
            if(!q_ok)
            {
                raw[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                q_max = fmaxf(q_max, __builtin_fabsf(raw[j][e]));
            }
        }
        float q_scale, q_back, k_back;
        odd = !power_to<true>(max_across_halves(q_max), 14, q_scale, q_back);
#pragma unroll
        for(int j = 0; j < CH; ++j)
        {
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                qf[j].pair(e, raw[2 * j + e / 2][2 * (e % 2)], raw[2 * j + e / 2][2 * (e % 2) + 1],
                        q_scale);
            }
        }
        float k_max = 0.0f, v_max = 0.0f;
#pragma unroll
        for(int i = 0; i < UPT; ++i)
        {
#pragma unroll
            for(int e = 0; e < 8; ++e)
            {
                k_max = fmaxf(k_max, __builtin_fabsf(k_raw[0][i][e / 4][e % 4]));
                v_max = fmaxf(v_max, __builtin_fabsf(v_raw[0][i][e]));
            }
        }
#pragma unroll
        for(int d = 1; d < 64; d *= 2)
        {
            k_max = fmaxf(k_max, __shfl_xor(k_max, d));
            v_max = fmaxf(v_max, __shfl_xor(v_max, d));
        }
        if(lane == 0)
        {
            first_max[2 * wave] = k_max;
            first_max[2 * wave + 1] = v_max;
        }
        __syncthreads();
#pragma unroll
        for(int w = 0; w < THREADS / 64; ++w)
        {
            k_max = fmaxf(k_max, first_max[2 * w]);
            v_max = fmaxf(v_max, first_max[2 * w + 1]);
        }
        // (the same in every lane; this makes the compiler see it, here and below)
        auto scalar = [](float x) __attribute__((always_inline)) -> float
        {
            return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
        };
        k_max = scalar(k_max);
        v_max = scalar(v_max);
        // (a step of zeros, padding in front, says nothing of what follows: K's as if
        // its largest were 8, which takes later keys up to 256; V's as if it were 2,
        // which takes up to 64 and eight of a channel down to 2^-12)
        odd = !power_to<true>(k_max == 0.0f ? 8.0f : k_max, 12, k_scale, k_back) || odd;
        odd = !power_to<false>(v_max == 0.0f ? 2.0f : v_max, 12, v_scale, v_back) || odd;
        k_scale = scalar(k_scale);
        v_scale = scalar(v_scale);
        v_back = scalar(v_back);
        if(v_src.rows_left < KEYS)
        {
            few_rows(0, v_goff);
        }
        qk_back = q_back * k_back;
        odd = odd || !(qk_back <= kX2Scores);
        if(__builtin_amdgcn_ballot_w64(odd && q_ok) != 0)
        {
            any_odd = 1;
        }
    }
    // item n of the 5 * UPT that split what was loaded: four pairs, then the store
    Split8 staged;
    auto store_pieces = [&](char *at, int piece_bytes, bool mine) __attribute__((always_inline))
    {
        if(UNITS % THREADS == 0 || mine)
        {
            *reinterpret_cast<u32x4 *>(at) = staged.h;
            *reinterpret_cast<u32x4 *>(at + piece_bytes) = staged.l;
        }
    };
    // Values of V that are too small for the pieces: the eight that a thread splits
    // together are a channel's, and all of them below 2^-2 once scaled but not all zeros.
    // (Otherwise what the pieces lose, 2^-25, is 2^-23 of the largest of the eight or
    // less, whatever the other channels and keys hold.)  large: some value was moved
    // to 2^13 or beyond.
    bool too_small = false, large = false;
    float unit_max = 0.0f;
    const float v_least = LEAST * v_back, v_large = 0x1p13f * v_back;
    auto look_at_pair = [&](int j, float a, float b) __attribute__((always_inline))
    {
        const float x = __builtin_fabsf(a), y = __builtin_fabsf(b);
        unit_max = j == 0 ? fmaxf(x, y) : max3(unit_max, x, y);
    };
    auto look_at_unit = [&]() __attribute__((always_inline))
    {
        too_small |= __builtin_amdgcn_ballot_w64(unit_max < v_least && unit_max > 0.0f) != 0;
        large |= __builtin_amdgcn_ballot_w64(unit_max >= v_large) != 0;
    };
    auto split_k = [&](int set, int n, char *lds_k) __attribute__((always_inline))
    {
        const int i = n / 5, j = n % 5;
        if(j < 4)
        {
            staged.pair(j, k_raw[set][i][j / 2][2 * (j % 2)], k_raw[set][i][j / 2][2 * (j % 2) + 1],
                    k_scale);
        }
        else
        {
            store_pieces(lds_k + k_at + k_lds(i), CH * 1024, i * THREADS + tid < UNITS);
        }
    };
    auto split_v = [&](int set, int n, char *lds_v) __attribute__((always_inline))
    {
        const int i = n / 5, j = n % 5;
        if(j < 4)
        {
            staged.pair(j, v_raw[set][i][2 * j], v_raw[set][i][2 * j + 1], v_scale);
            look_at_pair(j, v_raw[set][i][2 * j], v_raw[set][i][2 * j + 1]);
        }
        else
        {
            store_pieces(lds_v + v_at + v_lds(i), 2 * DB * 1024, i * THREADS + tid < UNITS);
            look_at_unit();
        }
    };
    // (chunk ch of a key is 32 * ch ^ the first one's place: bits below 512)
    int k_base = grp * GB + half * 512 + k_place(col, half) * 16;
    const int Vw = 2 * BUF + grp * GB + lane * 16;
    // c: from what m_run and the scores are in to powers of two
    // (1/sqrt(head) as two floats, and its product with log2(e) rounded once: what
    // the factors are off by, every row's sum and logsumexp are)
    constexpr double kScale = HEAD == 32 ? 0.17677669529663688 : HEAD == 64 ? 0.125 : 0.08838834764831845;
    constexpr float kScaleHi = (float)kScale, kScaleLo = (float)(kScale - (double)kScaleHi);
    constexpr float kScaleLog2e = (float)(kScale * 1.4426950408889634);
    static_assert(HEAD == 32 || HEAD == 64 || HEAD == 128, "kScale");
    float to_scores = kScaleHi * qk_back;
    float c = EXPLICIT ? kLog2e : kScaleLog2e * qk_back;
    float p_exp = (float)kX2PExp;       // the probabilities' power of two

    f32x16 o[DB];
#pragma unroll
    for(int db = 0; db < DB; ++db)
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            o[db][r] = 0.0f;
        }
    }
    float m_run = neg_inf(), l_run = 0.0f;

    // The operand fragments of a pass, in turn those of K (CH) and of V (2 * DB), each
    // read into one of two sets of registers while the other is in use.
    constexpr int FR = AHEAD_FR == 2 ? 4 : 2;
    Split8 fr[FR];
    auto read_k = [&](int buf, int ch) __attribute__((always_inline))
    {
        const char *at = lds + buf * BUF + ch * 1024 + (k_base ^ (32 * ch));
        fr[ch % FR].h = *reinterpret_cast<const u32x4 *>(at);
        fr[ch % FR].l = *reinterpret_cast<const u32x4 *>(at + CH * 1024);
    };
    auto read_v = [&](int buf, int n) __attribute__((always_inline))
    {
        const char *at = lds + Vw + buf * BUF + n * 1024;   // n: 16 keys n / DB, head block n % DB
        fr[(CH + n) % FR].h = *reinterpret_cast<const u32x4 *>(at);
        fr[(CH + n) % FR].l = *reinterpret_cast<const u32x4 *>(at + 2 * DB * 1024);
    };
    static_assert((CH + 2 * DB) % FR == 0 && CH >= AHEAD_FR && 2 * DB >= AHEAD_FR, "fragments in turn");
    // Scores of a step from K in buffer `buf`, its first fragment already read;
    // `between(t)` is called behind matrix instruction t of the NS, `last()` where
    // the first fragment of what follows can be read.
    auto scores = [&](int buf, f32x16 &s, auto between, auto last) __attribute__((always_inline))
    {
#pragma unroll
        for(int r = 0; r < 16; ++r)
        {
            s[r] = 0.0f;
        }
#pragma unroll
        for(int ch = 0; ch < CH; ++ch)
        {
            if(ch + AHEAD_FR < CH)
            {
                read_k(buf, ch + AHEAD_FR);
            }
            else
            {
                last(ch + AHEAD_FR - CH);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for(int n = 0; n < 3; ++n)
            {
                s = product(n, fr[ch % FR], qf[ch], s);
                between(3 * ch + n);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    Split8 pf[2];       // probabilities of 16 keys each
    // O^T += V^T P^T from V in buffer `buf`, likewise; NP instructions
    auto output = [&](int buf, auto between, auto last) __attribute__((always_inline))
    {
#pragma unroll
        for(int n = 0; n < 2 * DB; ++n)
        {
            if(n + AHEAD_FR < 2 * DB)
            {
                read_v(buf, n + AHEAD_FR);
            }
            else
            {
                last(n + AHEAD_FR - 2 * DB);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for(int t = 0; t < 3; ++t)
            {
                o[n % DB] = product(t, fr[(CH + n) % FR], pf[n / DB], o[n % DB]);
                between(3 * n + t);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // What hides keys of a step from this lane's query; register r holds key
    // 8 * (r / 4) + 4 * half + r % 4 of the wavefront's 32.
    auto apply_mask = [&](const StepSource &src, f32x16 &s) __attribute__((always_inline))
    {
        const int keys_here = src.rows_left - grp * kX2Rows;    // may be below 1
        if constexpr(EXPLICIT)
        {
            const int64_t mrow = my_row() * p.mask_ld + src.k_row0 + grp * kX2Rows;
            typedef f32x4 __attribute__((aligned(4))) f32x4_any;
            typedef uint32_t __attribute__((aligned(1))) u32_any;
            if(((not_open >> min(src.step + n_skip, 63)) & 1ull) == 0ull && keys_here >= kX2Rows)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    s[r] *= to_scores;
                }
            }
            else if(keys_here >= kX2Rows)
            {
                float madd[16];
#pragma unroll
                for(int rg = 0; rg < 4; ++rg)
                {
                    const int64_t at = mrow + 8 * rg + 4 * half;
                    if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                    {
                        const f32x4 v = *reinterpret_cast<const f32x4_any *>(
                                static_cast<const float *>(p.mask) + at);
#pragma unroll
                        for(int e = 0; e < 4; ++e)
                        {
                            madd[4 * rg + e] = v[e];
                        }
                    }
                    else
                    {
                        const uint32_t w = *reinterpret_cast<const u32_any *>(
                                static_cast<const uint8_t *>(p.mask) + at);
#pragma unroll
                        for(int e = 0; e < 4; ++e)
                        {
                            madd[4 * rg + e] = ((w >> (8 * e)) & 0xffu) != 0u ? 0.0f : neg_inf();
                        }
                    }
                }
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    s[r] = madd[r] == neg_inf() ? neg_inf() : s[r] * to_scores + madd[r];
                }
            }
            else
            {
                // a ragged step goes element by element: keys past its end are
                // hidden, their reads clamped to the row's last value
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    const int key = 8 * (r >> 2) + 4 * half + (r & 3);
                    const int64_t at = mrow + min(key, keys_here - 1);
                    float add;
                    if(MODE == NNTILE_HIP_MASK_ADDITIVE)
                    {
                        add = static_cast<const float *>(p.mask)[at];
                    }
                    else
                    {
                        add = static_cast<const uint8_t *>(p.mask)[at] != 0 ? 0.0f : neg_inf();
                    }
                    s[r] = (key >= keys_here || add == neg_inf()) ? neg_inf() : s[r] * to_scores + add;
                }
            }
        }
        else
        {
            const int64_t k_pos = src.k_pos + grp * kX2Rows;
            const bool diagonal = MODE == NNTILE_HIP_MASK_CAUSAL
                && k_pos + kX2Rows - 1 > wave_qpos_lo + p.causal_offset;
            if(keys_here < kX2Rows || diagonal)
            {
                const int64_t vis = MODE == NNTILE_HIP_MASK_CAUSAL
                    ? wave_qpos_lo + p.causal_offset - k_pos + col : (int64_t)kX2Rows;
                const int lim = (int)max((int64_t)-1, min(vis, (int64_t)keys_here - 1));
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    if(8 * (r >> 2) + 4 * half + (r & 3) > lim)
                    {
                        s[r] = neg_inf();
                    }
                }
            }
        }
    };
    // Online softmax in pieces: the maximum and what follows from it, then the
    // probabilities one by one.
    // (l_run is summed with its rounding errors kept: a wavefront of these forms adds
    // up to four times the steps that one of the fp32 kernel does)
    float mc = 0.0f, rs = 0.0f, l_low = 0.0f;
    auto softmax_head = [&](const f32x16 &s) __attribute__((always_inline))
    {
        float mx = neg_inf();
#pragma unroll
        for(int r = 0; r < 16; r += 2)
        {
            mx = max3(mx, s[r], s[r + 1]);
        }
        mx = max_across_halves(mx);
        const float m_new = fmaxf(m_run, mx);
        const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
        mc = m_use * c - p_exp;
        // the running maximum rarely moves after the first steps
        if(__builtin_amdgcn_ballot_w64(m_new != m_run) != 0)
        {
            const float alpha = fast_exp2((m_run - m_use) * c);
            l_run *= alpha;
            l_low *= alpha;
#pragma unroll
            for(int db = 0; db < DB; ++db)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    o[db][r] *= alpha;
                }
            }
            m_run = m_new;
        }
        rs = 0.0f;
        asm volatile("" : "+v"(mc));
    };
    auto softmax_one = [&](f32x16 &s, int r) __attribute__((always_inline))
    {
        float e = fast_exp2(fmaf(s[r], c, -mc));
        // (keeps the exponential where it is written, beside the matrix
        // instructions, instead of in front of its first use)
        asm volatile("" : "+v"(e));
        // (the one before: its exponential has arrived)
        if(r > 0)
        {
            rs += s[r - 1];
            asm volatile("" : "+v"(rs));
        }
        s[r] = e;
        if(r == 15)
        {
            const float add = (rs + e) - l_low, sum = l_run + add;
            l_low = (sum - l_run) - add;
            l_run = sum;
        }
    };
    // A long walk's output is put by and begun anew every PUT_BY steps.  Three
    // instructions a 16 keys round a sum that grows with the walk where a wavefront of
    // the fp32 kernel, eight keys an instruction, adds up a fourth of it: without this,
    // head 64, 16 x 2150 without a mask, A was off by 5.5e-7 against 5.2e-7 with fp32
    // products, 16 x 8192 10.4e-7 / 8.7e-7, and 8.5e-7 / 3.4e-7 where values have a mean of
    // 1; now 3.3e-7, 3.4e-7 and 1.0e-7.  In registers where they last, 16 steps (24 x 1750
    // 84.5 -> 85.5 us, 32 x 2150 causal 87.6 -> 88.7); else in scratch memory, which a full
    // chip writes and reads in 4 us: every 1024 keys of a wavefront where it walks all
    // of them (G = 1; head 128 without a mask, 16 x 4096 346 us without, 357 every 2048
    // keys, 366 every 1024, 386 every 512; 16 x 2150 141, 145, 152, 165; A there 5.9e-7,
    // 4.6e-7, 3.8e-7, with fp32 products 5.9e-7; values with a mean of 1 4.3e-7, 2.2e-7,
    // 1.3e-7, fp32 1.9e-7), else 2048.  In registers there: spills in the loop, 48 x 1024
    // 64 -> 73.  (Not carried in 1024 keys: head 128, values of one sign, 400 to 1100 keys of
    // a wavefront, up to 2.9e-7 where fp32 products have 1.4e-7.)
    constexpr bool BY_MEMORY = HEAD == 128 || (HEAD == 64 && (QW == 2 || EXPLICIT));
    constexpr int PUT_BY = !BY_MEMORY ? 16 : G == 1 ? 32 : 64;
    constexpr int PUT_BY_FP32 = BY_MEMORY ? 32 : 16;
    struct PutBy
    {
        f32x16 o[DB];
        float m;
    };
    PutBy put;
    float m_here = 0.0f;        // (of what is in memory, beside it where registers are short)
    float &m_by = EXPLICIT ? put.m : m_here;
    bool by = false;
    // (whoever might look at it there: the compiler keeps it out of registers)
    auto keep_in_memory = [&]() __attribute__((always_inline))
    {
        if(BY_MEMORY)
        {
            asm volatile("" : : "v"(&put) : "memory");
        }
    };
    auto add_what_was_put_by = [&]() __attribute__((always_inline))
    {
        keep_in_memory();
        const float m_use = (m_run == neg_inf()) ? 0.0f : m_run;
        const float alpha = fast_exp2((m_by - m_use) * c);
#pragma unroll
        for(int db = 0; db < DB; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o[db][r] = fmaf(put.o[db][r], alpha, o[db][r]);
            }
        }
    };
    auto put_by = [&]() __attribute__((always_inline))
    {
        if(by)
        {
            add_what_was_put_by();
        }
        by = true;
        m_by = m_run;
#pragma unroll
        for(int db = 0; db < DB; ++db)
        {
            put.o[db] = o[db];
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o[db][r] = 0.0f;
            }
        }
        keep_in_memory();
    };

    // ---- the walk -------------------------------------------------------------------
    if(n_steps > 0)
    {
#pragma unroll
        for(int n = 0; n < 5 * UPT; ++n)
        {
            split_k(0, n, lds);
        }
#pragma unroll
        for(int n = 0; n < 5 * UPT; ++n)
        {
            split_v(0, n, lds + 2 * BUF);
        }
        if(too_small)
        {
            any_odd = 1;
        }
        // K(1) and, with two sets, V(1) and K(2)
        advance(k_src);
        load_k(SETS - 1);
        if(SETS == 2)
        {
            advance(v_src);
            load_v(SETS - 1);
            advance(k_src);
            load_k(0);
        }
        __syncthreads();
    }
    // (one row that goes to fp32 from the start takes its workgroup with it; whoever
    // sets any_odd behind the walk has passed a barrier since)
    if(n_steps > 0 && __builtin_amdgcn_readfirstlane(any_odd) == 0)
    {
        // (steps past the last are that one again: nobody reads them)
        const int last_step = n_steps - 1;
        f32x16 s_even, s_odd;
        for(int n = 0; n < AHEAD_FR; ++n)
        {
            read_k(0, n);
        }
        scores(0, s_even, [](int) {}, [](int) {});
        apply_mask(s_src, s_even);
#pragma unroll
        for(int n = 0; n < 5 * UPT; ++n)
        {
            split_k(SETS - 1, n, lds + BUF);
        }
        advance(k_src);
        load_k(SETS - 1);
        __syncthreads();
        for(int n = 0; n < AHEAD_FR; ++n)
        {
            read_k(1, n);
        }
        // One pass; step i's scores are in s, those of step i+1 go into s_nxt.  The
        // barrier between the two parts: in front of it K(i+2) is written where K(i) was
        // read before the barrier of the last pass, and read behind it; behind it
        // V(i+1) is written where V(i-1) was read before it, and read behind the next.
        // Beside the scores: V's next rows are requested, the softmax of step i, the
        // pieces of its first 16 probabilities, K(i+2) into LDS.  Beside the output: K's
        // next rows are requested, V(i+1) into LDS.
        constexpr int NA = 1 + 16 + 4 + 5 * UPT;
        constexpr int NB = 5 * UPT;
        auto item_a = [&](int n, int buf, f32x16 &s) __attribute__((always_inline))
        {
            if(n == 0)
            {
                softmax_head(s);
            }
            else if(n < 17)
            {
                softmax_one(s, n - 1);
            }
            else if(n < 21)
            {
                const int j = n - 17;
                pf[0].pair(j, s[2 * j], s[2 * j + 1], kX2PPieces);
            }
            else
            {
                split_k(buf % SETS, n - 21, lds + buf * BUF);
            }
        };
        // the pieces of the other 16 probabilities
        auto pieces_b = [&](const f32x16 &s) __attribute__((always_inline))
        {
#pragma unroll
            for(int n = 0; n < 4; ++n)
            {
                pf[1].pair(n, s[8 + 2 * n], s[8 + 2 * n + 1], kX2PPieces);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto first_v = [&](int buf) __attribute__((always_inline))
        {
#pragma unroll
            for(int n = 0; n < AHEAD_FR; ++n)
            {
                read_v(buf, n);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // INNER: the rows to be requested are whole steps of the tiles that the last ones
        // requested are in: no branch, one instruction at a time behind the matrix
        // instructions.  (With a branch around each, or all at once, the wavefront
        // stands at its own loads: 32 x 4096, head 64, 264 and 241 us.)
        auto pass = [&](auto inner_tag, auto buf_tag, f32x16 &s, f32x16 &s_nxt)
            __attribute__((always_inline))
        {
            constexpr bool INNER = decltype(inner_tag)::value;
            constexpr int buf = decltype(buf_tag)::value;
            constexpr int v_set = SETS == 2 ? buf : 0, k_set = buf % SETS;
            if(SETS == 1)
            {
                // (the places of the other chunks are worked out again in each pass)
                asm volatile("" : "+v"(k_base));
            }
            // V(i+2) with two sets, V(i+1) with one
            if(INNER)
            {
                v_src.V += KEYS * HEAD;
            }
            else
            {
                advance(v_src);
                load_v(v_set);
            }
            scores(buf ^ 1, s_nxt, [&](int t) __attribute__((always_inline))
            {
#pragma unroll
                for(int n = 0; n < 8 * UPT; ++n)
                {
                    if(INNER && n >= t * 8 * UPT / NS && n < (t + 1) * 8 * UPT / NS)
                    {
                        load_v_piece(v_set, n);
                    }
                }
#pragma unroll
                for(int n = 0; n < NA; ++n)
                {
                    if(n >= t * NA / NS && n < (t + 1) * NA / NS)
                    {
                        item_a(n, buf, s);
                    }
                }
            }, [](int) {});
            __syncthreads();
            // (V(i) was written behind the last barrier: read behind this one, and
            // behind the reads what needs no operand)
            first_v(buf);
            pieces_b(s);
            // K(i+4) with two sets, K(i+3) with one
            if(INNER)
            {
                k_src.K += KEYS * HEAD;
            }
            else
            {
                advance(k_src);
                load_k(k_set);
            }
            output(buf, [&](int t) __attribute__((always_inline))
            {
#pragma unroll
                for(int n = 0; n < 2 * UPT; ++n)
                {
                    if(INNER && n >= t * 2 * UPT / NP && n < (t + 1) * 2 * UPT / NP)
                    {
                        load_k_piece(k_set, n);
                    }
                }
#pragma unroll
                for(int n = 0; n < NB; ++n)
                {
                    if(n >= t * NB / NP && n < (t + 1) * NB / NP)
                    {
                        split_v((buf ^ 1) % SETS, n, lds + (2 + (buf ^ 1)) * BUF);
                    }
                }
            }, [&](int n) __attribute__((always_inline)) { read_k(buf, n); });
            advance(s_src);
            apply_mask(s_src, s_nxt);
        };
        auto two_passes = [&](auto inner_tag) __attribute__((always_inline))
        {
            pass(inner_tag, std::integral_constant<int, 0>{}, s_even, s_odd);
            pass(inner_tag, std::integral_constant<int, 1>{}, s_odd, s_even);
        };
        // passes whose two steps of either request lie inside a tile, in pairs
        auto inner_pairs = [&](const StepSource &src) __attribute__((always_inline)) -> int
        {
            return (min(src.rows_left / KEYS, last_step - src.step + 1) - 1) / 2;
        };
        int pairs = last_step / 2, since = 0;
#pragma unroll 1
        while(pairs > 0)
        {
            const int inside_tile = min(inner_pairs(k_src), inner_pairs(v_src));
            const int inner = min(min(pairs, PUT_BY / 2 - since), inside_tile);
#pragma unroll 1
            for(int n = 0; n < inner; ++n)
            {
                two_passes(std::integral_constant<bool, true>{});
            }
            auto inside = [&](StepSource &src) __attribute__((always_inline))
            {
                src.step += 2 * inner;
                src.rows_left -= 2 * inner * KEYS;
                src.k_row0 += 2 * inner * KEYS;
                src.k_pos += 2 * inner * KEYS;
            };
            inside(k_src);
            inside(v_src);
            pairs -= inner;
            since += inner;
            if(pairs > 0 && inner == inside_tile)
            {
                two_passes(std::integral_constant<bool, false>{});
                --pairs;
                ++since;
            }
            if(pairs > 0 && since >= PUT_BY / 2)
            {
                put_by();
                since = 0;
            }
        }
        if(last_step & 1)
        {
            pass(std::integral_constant<bool, false>{}, std::integral_constant<int, 0>{}, s_even, s_odd);
            s_even = s_odd;
        }
        if(large)
        {
            any_large = 1;
        }
        __syncthreads();
#pragma unroll
        for(int n = 0; n < 21; ++n)
        {
            item_a(n, 0, s_even);
        }
        first_v(last_step & 1);
        pieces_b(s_even);
        output(last_step & 1, [](int) {}, [](int) {});
        if(by)
        {
            add_what_was_put_by();
        }
    }

    // ---- results that the pieces could not carry: once more in fp32 --------------------
    // (A row whose output, as a mean of scaled values, is below 2^-2 was taken from
    // values or of probabilities in the last bits of the pieces; where values of V come
    // up to 2^16, three bits above the others, the bound moves with them.)
    if(n_steps > 0)
    {
        float o_max = 0.0f, o_sum = 0.0f;
#pragma unroll
        for(int db = 0; db < DB; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o_max = fmaxf(o_max, __builtin_fabsf(o[db][r]));
                o_sum += o[db][r];
            }
        }
        o_max = max_across_halves(o_max);
        const float l_row = sum_across_halves(l_run);
        const float o_least = (any_large != 0 ? 0x1p1f : 0x1p-2f) * kX2PPieces * l_row;
        // (a NaN or an infinity among the outputs is one in their sum)
        odd = odd || !(l_row < __builtin_huge_valf())
            || !(__builtin_fabsf(o_sum) < __builtin_huge_valf())
            || (o_max > 0.0f && o_max < o_least);
        if(__builtin_amdgcn_ballot_w64(odd && q_ok) != 0 || too_small)
        {
            any_odd = 1;
        }
        __syncthreads();
        if(any_odd != 0)
        {
            qk_back = 1.0f;
            to_scores = kScaleHi;
            c = EXPLICIT ? kLog2e : kScaleLog2e;
            v_back = kX2PPieces;        // (undone below)
            p_exp = 0.0f;
            m_run = neg_inf();
            l_run = l_low = 0.0f;
            by = false;
#pragma unroll
            for(int db = 0; db < DB; ++db)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    o[db][r] = 0.0f;
                }
            }
            // Operands come from the caches, four groups of eight head values (two
            // halves of 16 bytes a lane) and eight keys ahead, the first of a step
            // during the products of the step before.
            constexpr int GROUPS = HEAD / 8, AHEAD = 4, KEYS_AHEAD = 8;
            const char *Q_at = reinterpret_cast<const char *>(Qt + my_row() * HEAD + 4 * half);
            f32x4 k_op[AHEAD], q_op[AHEAD];
            float v_op[KEYS_AHEAD][DB];
            auto read_kq = [&](const char *K_at, int g) __attribute__((always_inline))
            {
                k_op[g % AHEAD] = *reinterpret_cast<const f32x4 *>(K_at + 32 * g);
                q_op[g % AHEAD] = *reinterpret_cast<const f32x4 *>(Q_at + 32 * g);
            };
            // (rows past the end of the tile are its last one)
            auto keys_at = [&](const StepSource &src) __attribute__((always_inline)) -> const char *
            {
                return reinterpret_cast<const char *>(src.K)
                    + (uint32_t)((min(grp * kX2Rows + col, src.rows_left - 1) * HEAD + 4 * half) * 4);
            };
            auto read_value = [&](const StepSource &src, int r) __attribute__((always_inline))
            {
                const int key = grp * kX2Rows + 8 * (r >> 2) + 4 * half + (r & 3);
                const char *at = reinterpret_cast<const char *>(src.V)
                    + (uint32_t)((min(key, src.rows_left - 1) * HEAD + col) * 4);
#pragma unroll
                for(int db = 0; db < DB; ++db)
                {
                    v_op[r % KEYS_AHEAD][db] = *reinterpret_cast<const float *>(at + 128 * db);
                }
            };
            StepSource src = first_step();
            const char *K_at = keys_at(src);
#pragma unroll
            for(int g = 0; g < AHEAD; ++g)
            {
                read_kq(K_at, g);
            }
            // (keys behind the last that this wavefront's queries see are not walked)
#pragma unroll 1
            while(MODE != NNTILE_HIP_MASK_CAUSAL
                    || src.k_pos + grp * kX2Rows <= wave_qpos_lo + kX2Rows - 1 + p.causal_offset)
            {
                f32x16 s;
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    s[r] = 0.0f;
                }
#pragma unroll
                for(int g = 0; g < GROUPS; ++g)
                {
                    const f32x4 k = k_op[g % AHEAD], q = q_op[g % AHEAD];
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                    {
                        s = __builtin_amdgcn_mfma_f32_32x32x2f32(k[e], q[e], s, 0, 0, 0);
                    }
                    if(g + AHEAD < GROUPS)
                    {
                        read_kq(K_at, g + AHEAD);
                    }
                    else
                    {
                        read_value(src, 2 * (g + AHEAD - GROUPS));
                        read_value(src, 2 * (g + AHEAD - GROUPS) + 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                apply_mask(src, s);
                softmax_head(s);
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    softmax_one(s, r);
                }
                l_low = 0.0f;       // (of an infinite sum: NaN)
                StepSource next = src;
                advance(next);
                K_at = keys_at(next);
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
#pragma unroll
                    for(int db = 0; db < DB; ++db)
                    {
                        o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(v_op[r % KEYS_AHEAD][db], s[r], o[db], 0, 0, 0);
                    }
                    if(r + KEYS_AHEAD < 16)
                    {
                        read_value(src, r + KEYS_AHEAD);
                    }
                    else if(r >= 16 - AHEAD)
                    {
                        read_kq(K_at, r + AHEAD - 16);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if(src.step + 1 == n_steps)
                {
                    break;
                }
                if(src.step % PUT_BY_FP32 == PUT_BY_FP32 - 1)
                {
                    put_by();
                }
                src = next;
            }
            if(by)
            {
                add_what_was_put_by();
            }
        }
        if(!EXPLICIT && m_run != neg_inf())
        {
            const float m = m_run * qk_back;
            m_run = fmaf(m, kScaleHi, m * kScaleLo);        // the maximum of the scores
        }
        const float p_back = p_exp == 0.0f ? 1.0f : 0x1p-4f;
        l_run *= p_back;
        v_back *= p_back / kX2PPieces;
#pragma unroll
        for(int db = 0; db < DB; ++db)
        {
#pragma unroll
            for(int r = 0; r < 16; ++r)
            {
                o[db][r] *= v_back;
            }
        }
    }

    // ---- the key blocks' results into those of the first ---------------------------------
    if constexpr(G > 1)
    {
        // word w of lane l of wavefront (q, g > 0) sits at (((g-1)*QW + q)*NW + w)*64 + l
        constexpr int NW = 2 + 16 * DB;
        static_assert((G - 1) * QW * NW * 256 <= 4 * BUF, "exchange area does not fit");
        float *area = reinterpret_cast<float *>(lds);
        __syncthreads();        // everyone is done with the buffers
        if(grp > 0)
        {
            float *dst = area + ((grp - 1) * QW + qw) * NW * 64 + lane;
            dst[0] = m_run;
            dst[64] = l_run;
#pragma unroll
            for(int db = 0; db < DB; ++db)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    dst[(2 + 16 * db + r) * 64] = o[db][r];
                }
            }
        }
        __syncthreads();
        if(grp > 0)
        {
            return;
        }
#pragma unroll
        for(int v = 0; v < G - 1; ++v)
        {
            const float *src = area + (v * QW + qw) * NW * 64 + lane;
            const float m_other = src[0];
            const float m_new = fmaxf(m_run, m_other);
            const float m_use = (m_new == neg_inf()) ? 0.0f : m_new;
            const float a_mine = fast_exp2((m_run - m_use) * kLog2e);
            const float a_other = fast_exp2((m_other - m_use) * kLog2e);
            l_run = l_run * a_mine + src[64] * a_other;
#pragma unroll
            for(int db = 0; db < DB; ++db)
            {
#pragma unroll
                for(int r = 0; r < 16; ++r)
                {
                    o[db][r] = o[db][r] * a_mine + src[(2 + 16 * db + r) * 64] * a_other;
                }
            }
            m_run = m_new;
        }
    }

    // ---- epilogue ---------------------------------------------------------------------
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    // no visible key for this query (a NaN among its scores: as in the 16-bit kernel)
    const bool empty = l_tot == 0.0f;
    if constexpr(PARTS)
    {
        if(q_ok)
        {
            // (a sum that is NaN goes out as it is, with some finite maximum)
            const int64_t row = ((int64_t)part * p.batch + b) * p.q_seq + my_row();
            if(half == 0)
            {
                p.part_ml[2 * row] = empty ? neg_inf() : l_tot > 0.0f ? m_run : 0.0f;
                p.part_ml[2 * row + 1] = l_tot;
            }
            float *dst = p.part_o + row * HEAD + 4 * half;
#pragma unroll
            for(int db = 0; db < DB; ++db)
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
    if(!q_ok || !(l_tot > 0.0f || p.overwrite))
    {
        return;     // leave lse and A as they are
    }
    const float lse_new = empty ? neg_inf() : m_run + __logf(l_tot);
    float *lse_ptr = p.lse[q_tile0 + qt] + (int64_t)b * q_len + my_row();
    const float lse_old = p.overwrite ? neg_inf() : *lse_ptr;
    float w_old = 0.0f, w_new = 0.0f, lse_out = neg_inf();
    if(!empty)
    {
        merge_weights(lse_old, lse_new, w_old, w_new, lse_out);
    }
    if(half == 0)
    {
        *lse_ptr = lse_out;
    }
    const float w_o = empty ? 0.0f : w_new / l_tot;
    float *Arow = static_cast<float *>(p.A[q_tile0 + qt]) + ((int64_t)b * q_len + my_row()) * HEAD;
#pragma unroll
    for(int db = 0; db < DB; ++db)
    {
#pragma unroll
        for(int rg = 0; rg < 4; ++rg)
        {
            float *dst = Arow + db * 32 + 8 * rg + 4 * half;
            f32x4 v;
#pragma unroll
            for(int e = 0; e < 4; ++e)
            {
                v[e] = empty ? 0.0f : o[db][4 * rg + e] * w_o;
            }
            if(w_old != 0.0f)
            {
                const f32x4 old = *reinterpret_cast<const f32x4 *>(dst);
#pragma unroll
                for(int e = 0; e < 4; ++e)
                {
                    v[e] += w_old * old[e];
                }
            }
            *reinterpret_cast<f32x4 *>(dst) = v;
        }
    }
}

template<int HEAD, int QW, int G, bool PARTS = false>
static int launch_form(hipStream_t stream, PrefillParams &p, int mode)
{
    p.k_blocks_per_tile = (int)((p.k_tile + kX2Rows * G - 1) / (kX2Rows * G));
    p.q_blocks_per_tile = (int)((p.q_tile + kX2Rows * QW - 1) / (kX2Rows * QW));
    const int64_t n_wg = (int64_t)p.batch * p.n_slabs * p.n_q_tiles * p.q_blocks_per_tile
        * (PARTS ? p.n_parts : 1);
    if(n_wg <= 0 || n_wg > 0x7fffffff)
    {
        return NNTILE_HIP_EINVAL;
    }
    auto launch = [&](auto kernel) -> int
    {
        hipLaunchKernelGGL(kernel, dim3((unsigned)n_wg), dim3(64 * QW * G), 0, stream, p);
        return hipGetLastError() == hipSuccess ? NNTILE_HIP_OK : NNTILE_HIP_ELAUNCH;
    };
    if(mode == NNTILE_HIP_MASK_NONE)
    {
        return launch(sdpa_prefill_f16x2_kernel<HEAD, NNTILE_HIP_MASK_NONE, QW, G, PARTS>);
    }
    if(mode == NNTILE_HIP_MASK_CAUSAL)
    {
        return launch(sdpa_prefill_f16x2_kernel<HEAD, NNTILE_HIP_MASK_CAUSAL, QW, G, PARTS>);
    }
    if constexpr((QW * G == 4 || G == 4) && !PARTS)     // (masks given as values)
    {
        return mode == NNTILE_HIP_MASK_ADDITIVE
            ? launch(sdpa_prefill_f16x2_kernel<HEAD, NNTILE_HIP_MASK_ADDITIVE, QW, G>)
            : launch(sdpa_prefill_f16x2_kernel<HEAD, NNTILE_HIP_MASK_BOOL, QW, G>);
    }
    return NNTILE_HIP_EINVAL;
}

template<int HEAD>
static int launch_head(hipStream_t stream, PrefillParams &p, int mode, int form)
{
    if constexpr(HEAD == 64)
    {
        if(form == kF16x2Form24)
        {
            return launch_form<HEAD, 2, 4>(stream, p, mode);
        }
    }
    if constexpr(HEAD > 32)
    {
        if(form == kF16x2Form42)
        {
            return launch_form<HEAD, 4, 2>(stream, p, mode);
        }
        if(form == kF16x2Form81)
        {
            return launch_form<HEAD, 8, 1>(stream, p, mode);
        }
    }
    return form == kF16x2Form22 ? launch_form<HEAD, 2, 2>(stream, p, mode)
        : launch_form<HEAD, 4, 1>(stream, p, mode);
}

// Forms that take masks given as values: the small ones, and head 64's two by four
static bool with_values(int form)
{
    return form <= kF16x2Form41 || form == kF16x2Form24;
}

// The form that is expected to be done first; kF16x2None: the fp32 kernel's
// 32-query workgroups.
//
// A launch takes a fixed time (launch, prologue, epilogue), then the longer of two:
// the longest workgroup's walk, at the time of a pass when it has the CU to
// itself, and the passes that a CU gets, at the time a pass adds to a full one; a
// second and third round of workgroups start anew.  The times are fitted to
// launches of 1 to 200 heads of 64 to 8192 rows, causal and not, 4 to 8 % off in
// the mean; what the rule picks is within 1 to 2.5 % of the fastest of the first five
// in the mean.  us, the fp32 kernel's 32 queries / 22 / 41 / 42 / 81 - head 64, causal:
// 12 x 128 7.9 / 9.4 / 11.5 / 11.7 / 13.1; 12 x 1024 30 / 25 / 35 / 29 / 49; 48 x 1024
// 75 / 40.3 / 40.1 / 38.3 / 51; 200 x 1024 293 / 144 / 117 / 145 / 138; 12 x 4096 251 /
// 112 / 129 / 103 / 161; 32 x 4096 619 / 275 / 238 / 240 / 226.  Head 128, 48 x 1024: 177 /
// 90 / 67 / 63 / 75; without a mask 290 / 134 / 96 / 110 / 84; 32 x 4096 1490 / 648 / 432 /
// 444 / 386.
// Two query blocks and four key blocks (24, head 64: at 128 its pieces outgrow the LDS) are
// for launches of at most one such workgroup a CU, which 22 leaves with one wavefront on a
// SIMD: 22 / 24, causal, inputs of other calls in between, 12 x 1024 27.8 / 24.4, 6 x 2000 47.8 /
// 39.4, 4 x 4096 85 / 65.5, 2 x 8192 161 / 119, open 27.3 / 24.3, 47.3 / 40.2, 84 / 73.5, 160 /
// 136; two rounds of them, causal, 12 x 2000 50.7 / 42.1, 8 x 4096 94 / 82, but 32 x 1024 30.5 / 34.5.
// Errors against 64 bits: a wavefront's sums are half as long (A, 2-norm, 6 x 2000 open
// 4.0e-7 / 3.3e-7, values with a mean of 1 2.1e-7 / 1.2e-7; lse the same).
//
// Masks given as values: what they hide is not known in front of the launch.  A form is
// taken for its sum over three masks: open, causal, and a window, of which a workgroup
// walks its own rows and 64 keys more.  To look over more rows takes longer (scan).  us,
// the fp32 kernel / 22 / 41, open, causal, window of 32 either side - head 64: 2 x 800
// 30 29 12.5 / 30 28 18.5 / 40 40 23; 12 x 1000 54 38 18.7 / 39 38 23.4 / 53 53 27; 32 x
// 1024 99 68 32 / 51 39 27 / 52 53 29; 64 x 1024 190 121 59 / 92 64 47 / 79 60 38; head
// 128: 2 x 800 51 51 18 / 49 47 26 / 58 57 31; 32 x 1024 232 151 75 / 113 78 56 / 80 77 40.
// (257 to 512 workgroups of the fp32 kernel at head 64: a window is slower with 22,
// the others gain more.)
// 22 / 24, in the same order: 12 x 1024 37.8 36.7 22.4 / 33.7 32.3 23.4; 6 x 2000 70.2 64.5 32.3 /
// 60.8 58.6 34.4; 16 x 1000 41.8 39.5 25.0 / 37.6 36.2 25.4: a window loses a twentieth, the
// others gain a tenth.
int prefill_f16x2_form(const PrefillParams &p, int head, int mode)
{
    struct Cost
    {
        int form, rows, keys;
        double fixed, alone, full, round;      // us: launch, pass, pass on a full CU, round
        double scan;                            // us: a mask's rows beyond 32
    };
    static const Cost costs[3][6] = {
        {{kF16x2None, 32, 128, 4.5, 1.59, 1.25, 0.5, 0.0}, {kF16x2Form22, 64, 64, 6.6, 0.76, 0.58, 1.5, 1.5},
            {kF16x2Form41, 128, 32, 6.6, 0.77, 0.56, 1.5, 3.3}},
        {{kF16x2None, 32, 128, 5.1, 2.74, 2.50, 1.2, 0.0}, {kF16x2Form22, 64, 64, 7.7, 1.13, 1.00, 2.3, 1.5},
            {kF16x2Form41, 128, 32, 7.7, 0.90, 0.78, 2.6, 3.3}, {kF16x2Form42, 128, 64, 8.8, 1.31, 1.50, 7.0, 0.0},
            {kF16x2Form81, 256, 32, 8.2, 1.30, 1.40, 9.0, 0.0}, {kF16x2Form24, 64, 128, 9.2, 1.95, 1.95, 5.0, 1.5}},
        {{kF16x2None, 32, 128, 7.2, 5.23, 5.50, 5.0, 0.0}, {kF16x2Form22, 64, 64, 10.4, 2.17, 2.33, 8.7, 3.5},
            {kF16x2Form41, 128, 32, 9.4, 1.55, 1.31, 5.5, 4.5}, {kF16x2Form42, 128, 64, 12.2, 2.30, 2.75, 11.0, 0.0},
            {kF16x2Form81, 256, 32, 10.3, 2.00, 2.85, 0.0, 0.0}}};
    const bool values = mode == NNTILE_HIP_MASK_ADDITIVE || mode == NNTILE_HIP_MASK_BOOL;
    int best = kF16x2None;
    double least = 0.0;
    for(const Cost &f : costs[head == 128 ? 2 : head == 64 ? 1 : 0])
    {
        // (masks given as values: the small forms; two by four, the last of them, where one
        // of the other pieces' forms is faster than the fp32 kernel, which a window favours)
        if(f.rows == 0 || (values && (!with_values(f.form)
                        || (f.form == kF16x2Form24 && best == kF16x2None))))
        {
            continue;
        }
        const int64_t all = p.n_q_tiles * ((p.q_tile + f.rows - 1) / f.rows);     // query blocks
        auto per_cu = [&](int64_t n) { return (double)p.batch * p.n_slabs * n / 256.0; };
        auto start = [&](double wgs) { return f.fixed + f.round * (ceil(wgs) - 1.0); };
        auto passes = [&](int64_t keys)
        {
            return ceil((double)(keys < 1 ? 1 : keys < p.k_seq ? keys : p.k_seq) / f.keys);
        };
        // every query block walks `keys`
        auto alike = [&](int64_t keys)
        {
            const double wgs = per_cu(all);
            return start(wgs) + passes(keys) * (wgs <= 1.0 ? f.alone : ceil(wgs) * f.full);
        };
        // row q walks `before` + q + 1; the workgroups of rows that see no key end at once
        // (32 heads, 984 x 209, causal from the last key, head 64: 15.1 us with 41, which
        // was taken for their sake, 12.5 with the fp32 kernel)
        auto causal = [&](int64_t before)
        {
            const int64_t rows = before >= 0 ? p.q_seq : p.q_seq + before > 1 ? p.q_seq + before : 1;
            const int64_t from = before > 0 ? before : 0, seen = (rows + f.rows - 1) / f.rows;
            const double wgs = per_cu(before < 0 && seen < all ? seen : all);
            const double most = passes(from + rows);
            const double first = passes(from + (rows < f.rows ? rows : f.rows));
            const double shared = 0.5 * (most + first) * wgs * f.full + (wgs > 1.0 ? 0.5 * first * f.full : 0.0);
            return start(wgs) + (most * f.alone > shared ? most * f.alone : shared);
        };
        double t = values ? alike(p.k_seq) + causal(0) + alike(f.rows + 64) + 3.0 * f.scan
            : mode == NNTILE_HIP_MASK_CAUSAL ? causal(p.q_pos0 - p.k_pos0 + p.causal_offset)
            : alike(p.k_seq);
        // (a close call stays with the fp32 kernel)
        if(f.form == kF16x2None)
        {
            t *= 0.94;
        }
        if(f.form == kF16x2None || t < least)
        {
            best = f.form;
            least = t;
        }
    }
    return best;
}

int launch_prefill_f16x2_parts(hipStream_t stream, PrefillParams &p, int head, int mode)
{
    return head == 64 ? launch_form<64, 2, 2, true>(stream, p, mode)
        : head == 128 ? launch_form<128, 2, 2, true>(stream, p, mode) : NNTILE_HIP_EUNSUPPORTED;
}

int launch_prefill_f16x2(hipStream_t stream, PrefillParams &p, int head, int mode, int form)
{
    if(mode < NNTILE_HIP_MASK_ADDITIVE || mode > NNTILE_HIP_MASK_BOOL)
    {
        return NNTILE_HIP_EINVAL;
    }
    if(!with_values(form) && mode != NNTILE_HIP_MASK_NONE && mode != NNTILE_HIP_MASK_CAUSAL)
    {
        form = kF16x2Form41;
    }
    switch(head)
    {
        case 32:
            return launch_head<32>(stream, p, mode, form);
        case 64:
            return launch_head<64>(stream, p, mode, form);
        case 128:
            return launch_head<128>(stream, p, mode, form);
        default:
            return NNTILE_HIP_EUNSUPPORTED;
    }
}

} // namespace nntile_hip
