"""The pieces that a field is cut into for its transfer (pieceOf in tsp_transfer.h), against the field's own
addresses: records of one and several words, pieces that start inside a record, fields of more than 2^32 words."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <cstdio>
#include <initializer_list>
#include "tsp_transfer.h"
int main()
{
    using namespace tsp;
    long bad = 0, tested = 0;
    char* const dev = reinterpret_cast<char*>(1ull << 40);   // (addresses only: nothing is read)
    for (const uint64_t n : { 1ull, 7ull, 1000ull, (1ull << 31) * 3ull - 3ull, (1ull << 32) + 12345ull })
    {
        for (const uint32_t comps : { 1u, 2u, 3u })
        {
            for (const uint32_t stride : { 4u * comps, 16u })
            {
                const XferField f{ nullptr, dev, stride, comps, n };
                for (uint64_t k = 0; k < 40; k++)
                {
                    const uint64_t done = n * k / 40u;
                    const uint32_t words = static_cast<uint32_t>(std::min<uint64_t>(n - done, 5000u));
                    const XferPiece p = pieceOf(f, done, words, 77u);
                    for (uint32_t i = 0; i < words; i += words < 200u ? 1u : 97u)
                    {
                        // the kernel's address of word i of the piece (32-bit word numbers), and the field's
                        const uint32_t word = p.first + i, rec = word / p.comps;
                        const char* got = p.dev + static_cast<size_t>(rec) * p.stride + 4u * (word - rec * p.comps);
                        const uint64_t w = done + i;
                        const char* want = dev + (w / comps) * stride + 4u * (w % comps);
                        tested++;
                        bad += got != want || p.at != 77u || p.n != words;
                    }
                }
            }
        }
    }
    std::printf("tested %ld wrong %ld\n", tested, bad);
    return bad != 0 || tested == 0;
}
"""


def test_pieces_address_the_words_of_the_field(tmp_path):
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    inc = os.path.join(ROOT, "turbospharticles_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", inc, "-o", str(exe), str(src), "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
