"""How the workgroups of the down projection over listed neurons share the units that do not fill the chip once more (DownSplit of kernels_ffn_union.hip): every stage of every row
of every token tile comes to exactly one workgroup, under the number of a part of its own, and the launch that adds the parts sees as many.  The structs are compiled for the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOST = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#define __device__
#define __host__
#define __forceinline__ inline
constexpr int kGwM = 256, kGwBand = 8, kUnionParts = 4;
%s
int main(int argc, char ** argv) {
    const int rows = atoi(argv[1]), n_tiles = atoi(argv[2]), room = atoi(argv[3]), nr = rows / 128;         // (halves of units)
    int most = 0, before = 0;
    const int longest = room ? 512 : 0;
    for (int nk = 4; nk <= 512; nk += nk < 20 ? 1 : 7) {
        std::vector<unsigned char> seen((size_t)n_tiles * nr * nk, 0);
        std::vector<int> mask((size_t)n_tiles * nr, 0), parts((size_t)n_tiles * nr, 1);
        int split = 0;
        for (int b = 0; b < 256; ++b) {
            const DownSplit s(DownDeal(rows, n_tiles, room, b %% 8, b / 8, 32), longest, nk);
            if (s.parts < 1 || s.parts > (room ? kUnionParts : 1)) return 1;
            split = split || s.turns;
            for (int c = 0; c < s.count; ++c) {
                int ty, row0, n, part, of;
                s.unit(c, ty, row0, n, part, of);
                const int first = nk * part / of, stages = nk * (part + 1) / of - first;
                if (ty < 0 || ty >= n_tiles || row0 < 0 || row0 %% 128 || row0 + n > rows || part < 0 || part >= of || stages < 1 || first < 0 || first + stages > nk) return 2;
                if (of > 1 ? of != s.parts || c < s.deal.rounds : stages != nk) return 3;
                if (c + 4 < s.count && stages < 4) return 4;                // (as far ahead as copies go)
                for (int r = row0 / 128; r < (row0 + n) / 128; ++r) {
                    int & m = mask[(size_t)ty * nr + r];
                    if (m >> part & 1) return 5;
                    m |= 1 << part; parts[(size_t)ty * nr + r] = of;
                    for (int k = first; k < first + stages; ++k) if (seen[((size_t)ty * nr + r) * nk + k]++) return 6;
                }
            }
        }
        for (unsigned char v : seen) if (v != 1) return 7;
        for (size_t k = 0; k < mask.size(); ++k) if (mask[k] != (1 << parts[k]) - 1) return 8;
        for (int x = 0; x < 8; ++x) {                                       // the launch behind
            const DownDeal d(rows, n_tiles, room, x, 0, 32);
            const DownSplit s(d, longest, nk);
            if (s.parts > most) most = s.parts;
            for (int u = 0; u < d.rest; ++u) {
                int ty, row0;
                d.tile(d.rounds * d.slots + u, ty, row0);
                for (int r = row0 / 128; r < (row0 + kGwM) / 128; ++r) { int & p = parts[(size_t)ty * nr + r]; if (p != s.parts) return 9; p = 1; }
            }
        }
        for (int p : parts) if (p != 1) return 10;
        if (before && !split) return 11;                                    // what the longest list has not, no list has
        for (int x = 0; x < 8; ++x) {                                       // (and lists of few neurons never)
            const DownSplit s(DownDeal(rows, n_tiles, room, x, 0, 32), room ? 171 : 0, nk);
            if (s.turns) return 12;
        }
        before = split;
    }
    printf("%%d %%d\n", before, most);
    return 0;
}
"""


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    src = open(os.path.join(ROOT, "powerinfer_amd", "csrc", "kernels_ffn_union.hip")).read()
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text(HOST % src[src.index("struct DownDeal {"):src.index("// out[t][c] = sum over the listed neurons")])
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", str(d / "split"), str(d / "split.cpp")])
    return str(d / "split")


@pytest.mark.parametrize("rows", [256, 512, 768, 1024, 4096, 5120, 8192])
@pytest.mark.parametrize("n_tiles", [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 13, 14, 15, 16, 33])
@pytest.mark.parametrize("room", [0, 1])
def test_every_stage_once(rows, n_tiles, room, split):
    out = subprocess.run([split, str(rows), str(n_tiles), str(room)], timeout=60, capture_output=True, text=True)
    assert out.returncode == 0, out.returncode
    if (rows, n_tiles) in ((8192, 5), (5120, 8), (4096, 11), (8192, 6)):    # 20, 20, 22 and 24 units for 32 workgroups
        assert out.stdout.split() == (["1", "4" if n_tiles in (11, 6) else "3"] if room else ["0", "1"])
