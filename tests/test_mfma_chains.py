"""The chains of the 3D matrix-core adjoint (grid_mfma.hpp, ChainSlot and SlotList in
grid_tile.hpp), on the CPU.

* Plane sets: for every window width and start, each of the node's planes is in
  exactly one of the two 16-plane sets (at W = 14 a node can be in both, its planes
  split at 16), and the rule by which the accumulator registers of the second set are
  added to the planes gives every plane of the padded tile once.
* Slots: compiled for the host, ChainSlot's blocks cover the slot once for every
  instantiated layout, and for random tile rows the parts that the spread's rule
  writes are exactly those that SlotList lists for the fold, each carrying the sums
  of the chunks before it in its chain.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.parametrize("W", range(4, 15, 2))
def test_every_plane_in_one_set(W):
    P = 8 + W - 1
    off1, lo_max0 = max(0, P - 16), 16 - W
    sets2, dup = off1 > 0, lo_max0 + 1 < off1
    for lo in range(8):
        in1 = sets2 and lo > lo_max0
        in0 = not in1 or (dup and lo < off1)
        planes = []
        if in0:
            planes += [x for x in range(16) if lo <= x < lo + W]
        if in1:
            x_min = 16 - off1 if dup and in0 else 0
            planes += [x + off1 for x in range(x_min, 16) if lo <= x + off1 < lo + W]
        assert sorted(planes) == list(range(lo, lo + W)), (W, lo, planes)


@pytest.mark.parametrize("prec", ["single", "double"])
@pytest.mark.parametrize("W", range(4, 15, 2))
def test_set_sum(prec, W):
    P = 8 + W - 1
    off1 = max(0, P - 16)
    row = (lambda g, i: 4 * g + i) if prec == "single" else (lambda g, i: g + 4 * i)
    got = {}
    for g in range(4):
        for i in range(4):
            a = row(g, i)
            if a < P:
                terms = got.setdefault(a, [])
                terms.append(("set0", a))
                if off1 and prec == "single":
                    dg = -((i - off1 + 8) // 4 - 2)
                    rg = i - off1 + 4 * dg
                    if dg == 0:
                        terms.append(("set1", row(g, rg)))
                    elif g >= dg:
                        terms.append(("set1", row(g - dg, rg)))
                elif off1:
                    k = (off1 + 3) // 4
                    src, reg = (g - off1) & 3, i - k + 1 if g >= off1 - 4 * (k - 1) else i - k
                    if reg >= 0:
                        terms.append(("set1", row(src, reg)))
            if off1 and a + off1 >= 16:
                got.setdefault(a + off1, []).append(("set1", a))
    want = {a: ([("set0", a)] if a < 16 else []) + ([("set1", a - off1)] if off1 and 0 <= a - off1 < 16 else [])
            for a in range(P)}
    assert {a: sorted(t) for a, t in got.items()} == {a: sorted(t) for a, t in want.items()}


PROGRAM = r"""
#include "grid_tile.hpp"
#include <cstdio>
#include <random>
#include <set>
#include <vector>
using namespace cunfft;
static int bad = 0;
template <typename T, int W> void slot()
{
    using L = TileLayout<T, 3, W, 4, 0>;
    std::vector<int> hit(L::SC, 0);
    int cells = 0;
    for (int q0 = 0; q0 < L::Q0; ++q0)
        for (int q1 = 0; q1 < L::Q1; ++q1)
            for (int qL = 0; qL < L::QL; ++qL) {
                const int n = L::ext(8, L::P0, q0) * L::ext(8, L::P1, q1) * L::ext(8, L::PL, qL);
                const int o = ChainSlot<L>::off(q0, q1, qL);
                bad += qL == 0 && o % L::CPL != 0;
                bad += qL == 1 ? o + n > ChainSlot<L>::HALF1 : o < ChainSlot<L>::HALF1;
                for (int i = 0; i < n; ++i, ++cells)
                    if (o + i < 0 || o + i >= L::SC || hit[o + i]++) ++bad;
            }
    bad += cells != L::P0 * L::P1 * L::PL;
}
int main()
{
    slot<float, 4>(); slot<float, 6>(); slot<float, 8>(); slot<float, 10>(); slot<float, 12>(); slot<float, 14>();
    slot<double, 4>(); slot<double, 6>(); slot<double, 8>(); slot<double, 10>(); slot<double, 12>(); slot<double, 14>();
    std::mt19937 r(1);
    for (int rep = 0; rep < 3000; ++rep) {
        const int ntl = 1 + r() % 9, rows = 1 + r() % 4, sh = r() % 4;
        std::vector<uint32_t> nc(ntl * rows), c0(ntl * rows), tile;
        for (int t = 0; t < ntl * rows; ++t) {
            nc[t] = r() % 3 == 0 ? 0 : 1 + r() % (r() % 4 == 0 ? 20 : 2);
            c0[t] = tile.size();
            for (uint32_t k = 0; k < nc[t]; ++k) tile.push_back(t);
        }
        const uint32_t n = tile.size();
        // the spread's rule: cols[0] holds what the columns [0, 8) have gathered as
        // (chunk, column part), cols[1] the columns [8, 16)
        std::vector<std::set<std::pair<int, int>>> lo(n), hi(n);
        std::vector<int> wlo(n, 0), whi(n, 0);
        std::set<std::pair<int, int>> a0, a1;
        for (uint32_t c = 0; c < n; ++c) {
            a0.insert({(int)c, 0});
            a1.insert({(int)c, 1});
            const bool end = ((c + 1) & ((1u << sh) - 1)) == 0 || c + 1 >= n;
            const bool same = !end && tile[c + 1] == tile[c];
            const bool chain = !end && tile[c + 1] == tile[c] + 1 && tile[c + 1] % ntl != 0;
            if (same) continue;
            lo[c] = a0;
            wlo[c] = 1;
            if (chain) a0 = a1;
            else { hi[c] = a1; whi[c] = 1; a0.clear(); }
            a1.clear();
        }
        // the fold of every tile: each chunk's part 0 at its own tile and part 1 at the next
        for (int t = 0; t < ntl * rows; ++t) {
            const int row = t / ntl, l = t % ntl, prev = row * ntl + (l + ntl - 1) % ntl;
            std::set<std::pair<int, int>> sum;
            size_t terms = 0;
            const SlotList<true> s0(c0[t], nc[t], false, sh), s1(c0[prev], nc[prev], nc[t] > 0 && l > 0, sh);
            for (uint32_t k = 0; k < s0.n; ++k) {
                const uint32_t c = s0.at(k);
                if (c >= n || !wlo[c]) { ++bad; continue; }
                sum.insert(lo[c].begin(), lo[c].end());
                terms += lo[c].size();
            }
            for (uint32_t k = 0; k < s1.n; ++k) {
                const uint32_t c = s1.at(k);
                if (c >= n || !whi[c]) { ++bad; continue; }
                sum.insert(hi[c].begin(), hi[c].end());
                terms += hi[c].size();
            }
            std::set<std::pair<int, int>> want;
            for (uint32_t k = 0; k < nc[t]; ++k) want.insert({(int)(c0[t] + k), 0});
            for (uint32_t k = 0; k < nc[prev]; ++k) want.insert({(int)(c0[prev] + k), 1});
            bad += sum != want || terms != want.size();
        }
    }
    printf("bad %d\n", bad);
    return 0;
}
"""


def test_slots_and_lists(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.fail("hipcc is needed to compile the host replica")
    src, exe = tmp_path / "chains.cpp", tmp_path / "chains"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1",
                    "-I", os.path.join(ROOT, "include"),
                    "-I", os.environ.get("CSRC_DIR", os.path.join(ROOT, "cunfft_amd", "csrc")), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout == "bad 0\n"
