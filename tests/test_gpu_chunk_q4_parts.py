"""Products of transposed Q4_0 matrices whose tiles four workgroups share: the sums of one workgroup a tile, bit for bit, at edges of tiles and of parts, in every
tile and as the library chooses, with every epilogue; refused without room for the parts."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from powerinfer_amd import synth
from test_gpu_chunk_q4 import operand_layout

pytestmark = pytest.mark.gpu
TILES = [212, 213, 215, 223, 422, 423, 424, 433, 434]


@pytest.mark.parametrize("rows,cols", [(64, 1024), (192, 1280), (704, 1792), (128, 4352)])
def test_parts(rows, cols):
    L, rng = pl.init(), np.random.default_rng(rows + cols)
    q = synth.quantize_q4_0(rng.standard_normal((cols, rows)).astype(np.float32))
    dw = pl.DevBuf(host=np.concatenate([q.reshape(-1), np.zeros(16, np.uint8)]))
    for T in (1, 16, 17, 49, 130, 200):
        x, a1, a2 = rng.standard_normal((T, cols)).astype(np.float16), rng.standard_normal((T, rows)).astype(np.float32), rng.standard_normal((T, rows)).astype(np.float32)
        dx, d1, d2, dy = pl.DevBuf(host=operand_layout(x)), pl.DevBuf(host=a1), pl.DevBuf(host=a2), pl.DevBuf(T * rows * 4)
        bufs = [pl.DevBuf(host=np.full(T * rows, np.nan, np.float32)) for _ in range(6)]
        room = (C.c_void_p * 6)(*[b.ptr for b in bufs])

        def product(tile, epi, bufs):
            print(rows, cols, T, tile, epi, flush=True)
            rc = L.pi_k_gemm_q4_chunk_parts(dw.ptr, rows, cols, 1, dx.ptr, T, epi, d1.ptr if epi >= pl.EPI_ADD else None, d2.ptr if epi == pl.EPI_ADD2 else None, dy.ptr, tile, bufs, None)
            if rc != 0:
                return rc
            pl.sync()
            return dy.download(np.float32)

        for epi in (pl.EPI_NONE, pl.EPI_RELU, pl.EPI_ADD, pl.EPI_ADD2):
            want = product(212, epi, None)
            assert np.isfinite(want).all()
            for tile in [1000 + t for t in TILES] + [433, 0] if epi == pl.EPI_ADD else [1433, 0]:
                assert np.array_equal(product(tile, epi, room), want)
        assert product(1433, pl.EPI_NONE, None) != 0


def test_too_few_parts():
    L = pl.init()
    d = pl.DevBuf.zeros(1 << 20)
    room = (C.c_void_p * 6)(*[d.ptr] * 6)
    assert L.pi_k_gemm_q4_chunk_parts(d.ptr, 64, 768, 1, d.ptr, 3, 0, None, None, d.ptr, 1212, room, None) != 0
    assert L.pi_k_gemm_q4_chunk_parts(d.ptr, 64, 1024, 0, d.ptr, 3, 0, None, None, d.ptr, 1212, room, None) != 0
