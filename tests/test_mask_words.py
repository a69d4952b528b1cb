"""The words in which a scan of a mask is handed on (csrc/sdpa_mask_words.hpp),
compiled for the host: an entry is taken exactly where all its words are one
call's, and tags do not come again."""
import os
import subprocess

from nntile_amd import build as B

PROGRAM = r"""
#include <cstdio>
#include <random>
#include "sdpa_mask_words.hpp"
using nntile_hip::MaskWords;
#define CHECK(x) do { if(!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while(0)

int main()
{
    std::mt19937_64 rng(7);
    const uint64_t patterns[] = {0ull, ~0ull, 1ull, 1ull << 63, 0xff800000ff800000ull,
        0x3f8000003f800000ull, 0x00000000ffffffffull, 0xffffffff00000000ull};
    for(int trial = 0; trial < 2000; ++trial)
    {
        const uint64_t start = rng();
        uint64_t sets[2][2], w[2][5], open, hidden;
        for(auto &s : sets)
        {
            for(uint64_t &x : s)
            {
                x = trial % 2 ? patterns[rng() % 8] : rng();
            }
        }
        // the words of two calls that follow each other
        for(int c = 0; c < 2; ++c)
        {
            for(int i = 0; i < 5; ++i)
            {
                w[c][i] = MaskWords::word(i, MaskWords::tag(start, c), sets[c][0], sets[c][1]);
            }
            CHECK(MaskWords::take(w[c], MaskWords::tag(start, c), open, hidden));
            CHECK(open == sets[c][0] && hidden == sets[c][1]);
        }
        const uint64_t tag = MaskWords::tag(start, 1);
        // some words of the call before in place of this call's, or constants
        for(int mix = 1; mix < 32; ++mix)
        {
            for(int p = -1; p < 8; ++p)
            {
                uint64_t m[5];
                for(int i = 0; i < 5; ++i)
                {
                    m[i] = (mix >> i) & 1 ? (p < 0 ? w[0][i] : patterns[p]) : w[1][i];
                }
                CHECK(!MaskWords::take(m, tag, open, hidden));
            }
        }
        // one of the first four words with the right tag and other contents, the
        // other words right
        for(int i = 0; i < 4; ++i)
        {
            uint64_t m[5] = {w[1][0], w[1][1], w[1][2], w[1][3], w[1][4]};
            for(int bit = 0; bit < 32; ++bit)
            {
                m[i] = w[1][i] ^ (1ull << bit);
                CHECK(!MaskWords::take(m, tag, open, hidden));
            }
            m[i] = w[1][i] ^ (1ull + rng() % 0xffffffffull);
            CHECK(!MaskWords::take(m, tag, open, hidden));
        }
        // and beside a fifth word from before
        for(int i = 0; i < 4; ++i)
        {
            uint64_t m[5] = {w[1][0], w[1][1], w[1][2], w[1][3], w[0][4]};
            CHECK(!MaskWords::take(m, tag, open, hidden));
            m[i] = (tag << 32) | (rng() & 0xffffffffull);
            CHECK(!MaskWords::take(m, tag, open, hidden));
        }
        // tags: both halves differ between calls
        const uint64_t n = rng() % 0xffffffffull + 1ull;
        const uint64_t other = MaskWords::tag(start, n);
        CHECK((uint32_t)other != (uint32_t)MaskWords::tag(start, 0));
        CHECK((MaskWords::tag(start, 1) >> 32) != (MaskWords::tag(start, 0) >> 32));
    }
    std::puts("ok");
    return 0;
}
"""


def test_entries_are_taken_whole_or_not_at_all(tmp_path):
    src, exe = tmp_path / "words.cc", tmp_path / "words"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", B.CSRC, "-o", str(exe),
                    str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
