"""How the workgroups of the large-tile products share their units (WideDeal of gemm_wide.hpp): every row tile of every token tile comes to exactly one
workgroup, whole or as two halves, at shapes with long and short row tiles only, few tiles, many and none.  The struct is compiled for
the CPU, where a division by zero ends the program."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOST = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>
using std::max; using std::min;
#define __device__
#define __forceinline__ inline
struct Idx { unsigned x; };
static Idx blockIdx, gridDim;
%s
int main(int argc, char ** argv) {
    const int rows = atoi(argv[1]), n_tiles = atoi(argv[2]), band = atoi(argv[3]);
    std::vector<int> seen((size_t)n_tiles * rows);
    gridDim.x = wide_blocks((long long)n_tiles * ((rows + kGwM - 1) / kGwM));
    for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x) {
        const WideDeal d(rows, n_tiles, band);
        for (int c = 0; c < d.count; ++c) {
            int ty, row0, n;
            d.unit(c, ty, row0, n);
            if (ty < 0 || ty >= n_tiles || row0 < 0 || row0 %% (kGwM / 2) || n <= 0 || n > kGwM || row0 + n > rows) { printf("unit %%d %%d %%d\n", ty, row0, n); return 1; }
            for (int r = 0; r < n; ++r) ++seen[(size_t)ty * rows + row0 + r];
        }
    }
    for (int s : seen) if (s != 1) { printf("a row %%d times\n", s); return 2; }
    return 0;
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    src = open(os.path.join(ROOT, "powerinfer_amd", "csrc", "gemm_wide.hpp")).read()
    consts = re.search(r"constexpr int kGwM = .*", src).group(0).split(", kGwStages")[0] + ";"
    band = re.search(r"constexpr int kGwBand = .*", src).group(0)
    body = src[src.index("struct WideDeal {"):src.index("struct WidePlace")]
    d = tmp_path_factory.mktemp("deal")
    (d / "deal.cpp").write_text(HOST % "\n".join([consts, band, body]))
    subprocess.check_call(["g++", "-O0", "-std=c++17", "-o", str(d / "deal"), str(d / "deal.cpp")])
    return str(d / "deal")


@pytest.mark.parametrize("rows", [128, 129, 256, 300, 384, 512, 1408, 2816, 22016])
@pytest.mark.parametrize("n_tiles", [1, 3, 8, 16, 130])
@pytest.mark.parametrize("band", [1, 8])
def test_every_unit_once(rows, n_tiles, band, deal):
    r = subprocess.run([deal, str(rows), str(n_tiles), str(band)], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, (r.returncode, r.stdout)


def test_no_tiles(deal):
    assert subprocess.run([deal, "1408", "0", "1"], timeout=30).returncode == 0
