// The words in which the workgroups that scan a mask for a whole launch hand on
// what they found, through memory that the caller lends for it and whose contents
// before are anybody's.  Plain C++, for the device and for a test on the host.
#pragma once

#include <cstdint>

#if defined(__HIP__)
#define NNTILE_MASK_WORDS_FN __host__ __device__ __forceinline__
#else
#define NNTILE_MASK_WORDS_FN inline
#endif

namespace nntile_hip
{

// Five words, stored and read without any order among them:
//   0, 1  lower and upper half of not_open, 2, 3 of not_hidden, each below the
//         lower 32 bits of the tag;
//   4     the whole tag ^ not_open ^ (not_hidden, halves exchanged).
// A reader takes them only where all five fit together, so that what was in memory
// before - it can stand in for some of them while the others have arrived - is not
// mistaken for an answer:
//   - one of the first four, beside the right fifth: a half of one set shares its half
//     of the fifth word with a half of the other set, which is the right one, so a
//     wrong one does not fit, whatever its tag;
//   - two or more of them beside the right fifth: each has to hold 32 bits of the tag;
//   - any of them beside a fifth word from before: that has to be the one value of 2^64
//     that goes with them.
// Tags differ from call to call in both halves, so words of earlier calls are like any
// others.  (Four words of which each was taken by itself, under a tag of 32 bits: any
// one that happened to be there was the answer for its half of a set, once in 2^32.)
struct MaskWords
{
    static constexpr int N = 5;

    static NNTILE_MASK_WORDS_FN uint64_t word(int i, uint64_t tag, uint64_t not_open,
            uint64_t not_hidden)
    {
        const uint64_t set = (i & 2) ? not_hidden : not_open;
        const uint64_t half = (i & 1) ? set >> 32 : set & 0xffffffffull;
        return i == 4 ? tag ^ not_open ^ ((not_hidden << 32) | (not_hidden >> 32))
            : (tag << 32) | half;
    }

    // Whether a word carries its part of the tag, where it has one of its own
    static NNTILE_MASK_WORDS_FN bool tagged(int i, uint64_t w, uint64_t tag)
    {
        return i == 4 || (uint32_t)(w >> 32) == (uint32_t)tag;
    }

    // What a word contributes to the sum (exclusive or) of an entry, which is zero
    // where the words fit together
    static NNTILE_MASK_WORDS_FN uint64_t share(int i, uint64_t w, uint64_t tag)
    {
        const uint64_t half = w & 0xffffffffull;
        return i == 4 ? w ^ tag : (i == 1 || i == 2) ? half << 32 : half;
    }

    // The sets of an entry, and whether it is that of the tag.
    static NNTILE_MASK_WORDS_FN bool take(const uint64_t (&w)[N], uint64_t tag,
            uint64_t &not_open, uint64_t &not_hidden)
    {
        not_open = (w[0] & 0xffffffffull) | (w[1] << 32);
        not_hidden = (w[2] & 0xffffffffull) | (w[3] << 32);
        bool ok = true;
        uint64_t sum = 0u;
        for(int i = 0; i < N; ++i)
        {
            ok = ok && tagged(i, w[i], tag);
            sum ^= share(i, w[i], tag);
        }
        return ok && sum == 0u;
    }

    // Tag of the n-th call of a process that started from a random number: an odd
    // step, so that 2^64 calls have different tags, whose lower half is odd too, so
    // that 2^32 calls have different lower halves.
    static NNTILE_MASK_WORDS_FN uint64_t tag(uint64_t start, uint64_t n)
    {
        return start + n * 0x9e3779b97f4a7c15ull;   // 2^64 over the golden ratio
    }
};

} // namespace nntile_hip
