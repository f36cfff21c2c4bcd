"""Which tiles the experts' products go in (pi_k_expert_tile), on the CPU: by the rows an expert has, the size of the matrices, and what a tile can address."""
import pytest

from powerinfer_amd import lib as pl


@pytest.mark.parametrize("experts,up,down,want", [
    (64, (1408, 4096), (4096, 1408), (128, 128, 128, 256)),          # 1.5 GB
    (8, (8192, 4096), (4096, 4096), (128, 128, 128, 256)),
    (16, (2816, 2048), (2048, 1408), (64, 128, 128, 128)),           # 276 MB
    (64, (128, 65536), (65536, 128), (64, 128, 128, 128)),           # too few rows for the large tiles
    (2, (32768, 65536), (65536, 16384), (128, 128, 128, 128)),       # 2^31 values of an expert: no tiles of 256 tokens
    (2, (16384, 16384), (65536, 32768), (128, 128, 128, 128)),
    (2, (32767, 65536), (65536, 16384), (128, 128, 128, 256)),
])
def test_by_rows_and_sizes(experts, up, down, want):
    tile = pl.load().pi_k_expert_tile
    assert tuple(tile(n * experts + more, experts, *up, *down) for n, more in ((52, 0), (52, 1), (132, 0), (132, 1))) == want
