"""The chunk rule and the XCD groups of the tile-staging kernels, on the CPU.

Compiled for the host from cunfft_amd/csrc/bin.hpp:

* ``chunk_shift`` / ``chunks_of``: a tile's chunks hold 2^base .. 256 nodes, fewer
  than 1 << kTileChunksLog of them until they are 256 long, and never more than
  c / 2^base rounded up, so a binning's ntiles + ceil(M / 2^base) chunk records
  suffice;
* ``xcd_chunk`` with ``xcd_group``: every chunk exactly once within the workgroups
  that ``xcd_grid`` launches, and from 64 chunks on the XCDs' shares differ by at
  most one group, an eighth of an XCD's share or less.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "bin.hpp"
#include <cstdio>
#include <vector>
using namespace cunfft;
int main()
{
    int bad = 0;
    for (int base = kChunkShiftMin; base <= kChunkShift; ++base)
        for (uint32_t c = 0; c < 20000; ++c) {
            const int s = chunk_shift(c, base);
            const uint32_t k = chunks_of(c, base), len = 1u << s;
            bad += !(s >= base && s <= kChunkShift);
            bad += !(k * (uint64_t)len >= c && (k == 0 ? c == 0 : (k - 1) * (uint64_t)len < c));
            bad += !(k <= (c + (1u << base) - 1) >> base);
            bad += !(s == kChunkShift || c >> s < 1u << kTileChunksLog);
            bad += !(s == base || c >> (s - 1) >= 1u << kTileChunksLog);   // no longer than needed
        }
    printf("chunks %d\n", bad);
    bad = 0;
    const uint32_t ns[] = {0, 1, 7, 8, 63, 64, 65, 127, 128, 129, 304, 511, 512, 1000, 1025,
                           4095, 4096, 8191, 8192, 8193, 41856};
    for (uint32_t n : ns)
        for (uint32_t more = 0; more < 20; more += 3) {
            const uint32_t g = xcd_group(n);
            std::vector<int> hit(n, 0);
            uint32_t on[kXcds] = {};
            const unsigned grid = xcd_grid((int64_t)n + more);
            for (unsigned b = 0; b < grid; ++b) {
                const int64_t c = xcd_chunk(b, n, g);
                if (c < 0) continue;
                if (c >= (int64_t)n) { ++bad; continue; }
                ++hit[c];
                ++on[b % kXcds];
            }
            for (uint32_t c = 0; c < n; ++c) bad += hit[c] != 1;
            uint32_t lo = n, hi = 0;
            for (uint32_t v : on) { lo = v < lo ? v : lo; hi = v > hi ? v : hi; }
            if (n >= 64) bad += hi - lo > g || 8 * g > n / kXcds;
        }
    printf("groups %d\n", bad);
    return 0;
}
"""


def test_chunks_and_xcd_groups(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.fail("hipcc is needed to compile the host replica")
    src, exe = tmp_path / "chunks.cpp", tmp_path / "chunks"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2",
                    "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "cunfft_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert out.split("\n")[:2] == ["chunks 0", "groups 0"], out
