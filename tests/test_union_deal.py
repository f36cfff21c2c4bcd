"""How the workgroups of the down projection over listed neurons share its units (DownDeal of kernels_ffn_union.hip): every part of every row of every token tile comes to
exactly one workgroup, and the sums behind it see the units that were shared.  The struct is compiled for the CPU."""
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
    const int rows = atoi(argv[1]), n_tiles = atoi(argv[2]), room = atoi(argv[3]);
    std::vector<int> seen((size_t)n_tiles * rows, 0), of((size_t)n_tiles * rows, 0);
    for (int b = 0; b < 256; ++b) {
        const DownDeal d(rows, n_tiles, room, b %% 8, b / 8, 32);
        for (int c = 0; c < d.count; ++c) {
            int ty, row0, n, part, parts;
            d.unit(c, ty, row0, n, part, parts);
            if (ty < 0 || ty >= n_tiles || row0 < 0 || row0 %% 128 || row0 + n > rows || part < 0 || part >= parts || parts > kUnionParts || (!room && parts > 1)) return 1;
            if (c + 1 < d.count && (parts > 1 || n != kGwM)) return 2;
            for (int r = row0; r < row0 + n; ++r) { int & s = seen[(size_t)ty * rows + r]; if (s >> part & 1) return 3; s |= 1 << part; of[(size_t)ty * rows + r] = parts; }
        }
    }
    for (size_t k = 0; k < seen.size(); ++k) if (of[k] < 1 || seen[k] != (1 << of[k]) - 1) return 4;
    for (int x = 0; x < 8; ++x) {
        const DownDeal d(rows, n_tiles, room, x, 0, 32);
        for (int u = 0; d.parts > 1 && u < d.rest; ++u) {
            int ty, row0;
            d.tile(d.rounds * d.slots + u, ty, row0);
            for (int r = row0; r < row0 + kGwM; ++r) { int & s = of[(size_t)ty * rows + r]; if (s != d.parts) return 5; s = 1; }
        }
    }
    for (int s : of) if (s != 1) return 6;
    return 0;
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    src = open(os.path.join(ROOT, "powerinfer_amd", "csrc", "kernels_ffn_union.hip")).read()
    d = tmp_path_factory.mktemp("deal")
    (d / "deal.cpp").write_text(HOST % src[src.index("struct DownDeal {"):src.index("// out[t][c] = sum over the listed neurons")])
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-o", str(d / "deal"), str(d / "deal.cpp")])
    return str(d / "deal")


@pytest.mark.parametrize("rows", [256, 512, 768, 1024, 4096, 5120, 8192])
@pytest.mark.parametrize("n_tiles", [1, 2, 3, 4, 7, 8, 15, 16, 33])
@pytest.mark.parametrize("room", [0, 1])
def test_every_part_once(rows, n_tiles, room, deal):
    assert subprocess.run([deal, str(rows), str(n_tiles), str(room)], timeout=30).returncode == 0
