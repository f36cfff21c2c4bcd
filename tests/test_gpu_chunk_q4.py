"""Prompt chunks straight from Q4_0 blocks: the products against float64 at edges of tiles, every tile against every other, and the operand layout's forms
of what they read, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from powerinfer_amd import synth

pytestmark = pytest.mark.gpu
TILES = {0: [112, 122, 123, 215, 232, 314, 323, 333, 334, 414, 423, 424, 434, 444, 624], 1: [212, 213, 215, 223, 422, 423, 424, 434]}


def operand_layout(x):
    """[T, cols] -> 16 tokens by 16, eight columns of a token in a row; tokens past T are NaN (read, and of no consequence)."""
    T, cols = x.shape
    full = np.full(((T + 15) // 16 * 16, cols), np.nan, np.float16)
    full[:T] = x
    return np.ascontiguousarray(full.reshape(-1, 16, cols // 8, 8).transpose(0, 2, 1, 3))


def row_layout(o, T, cols):
    return o.reshape(-1, cols // 8, 16, 8).transpose(0, 2, 1, 3).reshape(-1, cols)[:T]


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("rows,cols", [(64, 256), (192, 512), (704, 1280), (1088, 768)])
def test_products_from_blocks(rows, cols, trans):
    """Every tile at 1 .. 250 tokens, epilogues, W on 4 bytes only.  Bound: fp32 sums of n products, in parts of at most n terms, are within n * 2^-24 times
    the sum of the products' magnitudes of the exact sum of the same fp16 values (one more rounding per residual)."""
    L = pl.init()
    rng = np.random.default_rng(rows + cols + trans)
    w = rng.standard_normal((cols, rows) if trans else (rows, cols)).astype(np.float32)
    w[:, :32] = 0                                                   # blocks without a scale
    q = synth.quantize_q4_0(w)
    values = synth.dequantize_q4_0(q, w.shape[1]).reshape(w.shape).astype(np.float16).astype(np.float64)
    if trans:
        values = values.T
    for T, shift in ((1, 0), (16, 4), (17, 0), (49, 8), (130, 0), (250, 12)):
        x = rng.standard_normal((T, cols)).astype(np.float16)
        a1, a2 = (rng.standard_normal((T, rows)).astype(np.float32) for _ in range(2))
        dw = pl.DevBuf(host=np.concatenate([np.zeros(shift, np.uint8), q.reshape(-1), np.zeros(16, np.uint8)]))
        dx, d1, d2, dy = pl.DevBuf(host=operand_layout(x)), pl.DevBuf(host=a1), pl.DevBuf(host=a2), pl.DevBuf(T * rows * 4)
        want, size = x.astype(np.float64) @ values.T, np.abs(x.astype(np.float64)) @ np.abs(values.T)
        first = None
        for tile in TILES[trans] + [0]:
            print(rows, cols, trans, T, shift, tile, flush=True)
            pl.check(L.pi_k_gemm_q4_chunk(dw.ptr + shift, rows, cols, trans, dx.ptr, T, pl.EPI_NONE, None, None, dy.ptr, tile, None))
            pl.sync()
            got = dy.download(np.float32).reshape(T, rows)
            assert (np.abs(got - want) <= cols * 2.0 ** -24 * size).all()
            assert first is None or np.array_equal(got, first)      # one order of sums in every tile
            first = got
        for epi, add in ((pl.EPI_RELU, None), (pl.EPI_ADD, a1), (pl.EPI_ADD2, a1)):
            pl.check(L.pi_k_gemm_q4_chunk(dw.ptr + shift, rows, cols, trans, dx.ptr, T, epi, d1.ptr if add is not None else None, d2.ptr if epi == pl.EPI_ADD2 else None, dy.ptr, 0, None))
            pl.sync()
            y = np.maximum(first, 0) if add is None else first + a1
            assert np.array_equal(dy.download(np.float32).reshape(T, rows), y + a2 if epi == pl.EPI_ADD2 else y)


def test_sums_do_not_depend_on_the_number_of_tokens():
    """The first tokens of 512 have the bits they have alone."""
    L = pl.init()
    rng = np.random.default_rng(1)
    rows, cols = 2048, 1024
    for trans in (0, 1):
        q = synth.quantize_q4_0(rng.standard_normal((cols, rows) if trans else (rows, cols)).astype(np.float32))
        x, dw, out = rng.standard_normal((512, cols)).astype(np.float16), pl.DevBuf(host=q), {}
        for T in (5, 33, 200, 512):
            dx, dy = pl.DevBuf(host=operand_layout(x[:T])), pl.DevBuf(T * rows * 4)
            pl.check(L.pi_k_gemm_q4_chunk(dw.ptr, rows, cols, trans, dx.ptr, T, pl.EPI_NONE, None, None, dy.ptr, 0, None))
            pl.sync()
            out[T] = dy.download(np.float32).reshape(T, rows)
        assert all(np.array_equal(out[T], out[512][:T]) for T in out)


def test_what_the_products_refuse():
    L = pl.init()
    d = pl.DevBuf(1 << 20)
    call = lambda rows=64, cols=256, w=d.ptr, T=3, epi=0, add=None, tile=0: L.pi_k_gemm_q4_chunk(w, rows, cols, 0, d.ptr, T, epi, add, None, d.ptr, tile, None)  # noqa: E731
    assert call(rows=32) != 0 and call(cols=128) != 0 and call(w=d.ptr + 2) != 0 and call(T=0) != 0 and call(epi=pl.EPI_ADD) != 0 and call(tile=111) != 0
    assert L.pi_k_gemm_q4_chunk_supported(12288, 4096) and not L.pi_k_gemm_q4_chunk_supported(96, 4096) and not L.pi_k_gemm_q4_chunk_supported(1 << 20, 4096)


@pytest.mark.parametrize("T,cols,off", [(1, 32, 0), (17, 96, 0), (33, 4096, 0), (20, 8192, 0), (18, 4096, 4)])
def test_inputs_in_the_operand_layout(T, cols, off):
    """Norms into Q8_0 values: the operand layout holds what the row layout does, beside a plain copy by rows; norm weights off 16 bytes take the other kernel."""
    L = pl.init()
    rng = np.random.default_rng(cols)
    x = (3 * rng.standard_normal((T, cols))).astype(np.float32)
    nw, nb = ((rng.random(cols + 4) + 0.5).astype(np.float32) for _ in range(2))
    dx, dw, db = pl.DevBuf(host=x), pl.DevBuf(host=nw), pl.DevBuf(host=nb)
    slots = (T + 15) // 16 * 16
    for kind in (0, 1, 2):
        norm = pl.Norm(kind, 1e-5, dw.ptr + off if kind else None, db.ptr + off if kind == 2 else None)
        a, p, b, r = (pl.DevBuf(n * cols * 2) for n in (T, T, slots, T))
        pl.check(L.pi_k_norm_q8_round_f16(dx.ptr, T, cols, C.byref(norm), a.ptr, p.ptr, None))
        pl.check(L.pi_k_norm_q8_round_f16_ol(dx.ptr, T, cols, C.byref(norm), b.ptr, r.ptr, None))
        pl.sync()
        assert np.array_equal(row_layout(b.download(np.float16), T, cols), a.download(np.float16).reshape(T, cols))
        assert np.array_equal(r.download(np.float16), p.download(np.float16)) and np.array_equal(p.download(np.float16).reshape(T, cols), x.astype(np.float16))


@pytest.mark.parametrize("T,ff", [(1, 64), (17, 192), (130, 11008)])
def test_hidden_vectors_in_the_operand_layout(T, ff):
    """h through Q8_0 blocks, both layouts, and operands off 16 bytes (the other kernel), bit for bit."""
    L = pl.init()
    rng = np.random.default_rng(ff)
    u, g, l = (np.concatenate([rng.standard_normal(T * ff), np.zeros(4)]).astype(np.float32) for _ in range(3))
    l[5] = np.nan                                                   # counts as active, as in the sparse operators
    du, dg, dl = pl.DevBuf(host=u), pl.DevBuf(host=g), pl.DevBuf(host=l)
    odd = pl.DevBuf(host=np.concatenate([np.zeros(1, np.float32), u]))
    for gate in (dg.ptr, None):
        a, b, c = pl.DevBuf(T * ff * 2), pl.DevBuf(T * ff * 2), pl.DevBuf((T + 15) // 16 * 16 * ff * 2)
        pl.check(L.pi_k_ffn_h_q8_f16(du.ptr, gate, dl.ptr, 0.1, T, ff, a.ptr, None))
        pl.check(L.pi_k_ffn_h_q8_f16(odd.ptr + 4, gate, dl.ptr, 0.1, T, ff, b.ptr, None))
        pl.check(L.pi_k_ffn_h_q8_f16_ol(du.ptr, gate, dl.ptr, 0.1, T, ff, c.ptr, None))
        pl.sync()
        want = a.download(np.float16)
        assert np.array_equal(b.download(np.float16), want) and np.array_equal(row_layout(c.download(np.float16), T, ff), want.reshape(T, ff))
        assert want.any() and not want.all()
    assert L.pi_k_ffn_h_q8_f16_ol(odd.ptr + 4, None, dl.ptr, 0.1, T, ff, c.ptr, None) != 0
