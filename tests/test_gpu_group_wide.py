"""The grouped product's large tiles (256 rows x 128 tokens, group_wide_kernel): bit for bit the small tiles' results, whose order of sums
it keeps, and within bf16's rounding of float64, at the edges of tiles, halves of tiles, stages and units."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_latent_ops import dev, fetch, group_args, i32, rounded, store

pytestmark = pytest.mark.gpu


def run(g, tile, n, ldy, y_f32):
    y = pl.DevBuf.zeros(4 * n * ldy + 64)
    g.y = y.ptr
    pl.check(pl.init().pi_k_group_gemm_tile(C.byref(g), tile, None))
    pl.sync()
    got = y.download(np.uint32 if y_f32 else np.uint16)
    assert not got[n * ldy:].any()                                            # nothing behind the last row
    return got[:n * ldy].reshape(n, ldy), fetch(y, pl.F32 if y_f32 else pl.BF16, (n, ldy))


def same(a, b, y_f32):
    """Equal, and where the order of a float's operations is the compiler's (the GLU's), within one unit of the last place."""
    assert np.abs(a.astype(np.int64) - b.astype(np.int64)).max() <= 1


@pytest.mark.parametrize("rows,cols,kind,y_f32", [(129 + 7, 256, "plain", 0), (256, 320, "relu2", 0), (264, 256, "plain", 1), (384, 512, "glu", 0), (392, 256, "relu2", 0),
                                                  (270, 256, "plain", 0), (528, 384, "glu", 0), (400, 256, "pair", 0), (300, 256, "glu", 0)])
def test_experts_of_uneven_size(rows, cols, kind, y_f32):
    rng = np.random.default_rng(rows + cols)
    counts = [0, 1, 16, 63, 64, 65, 127, 128, 129, 300, 0, 193]
    E, n, div = len(counts), sum(counts), 3
    T = (n + div - 1) // div
    W = rounded(rng.standard_normal((E, rows, cols)) / np.sqrt(cols))
    x = rounded(rng.standard_normal((T, cols)))
    perm = rng.permutation(T * div)[:n].astype(np.int32)
    pw = rng.random(T * div).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(counts)])
    glu = kind in ("glu", "pair")
    ldy = ((rows // 2 if glu else rows) + 7) // 8 * 8
    bufs = [store(W.reshape(-1, cols), pl.BF16), store(x, pl.BF16), i32(off), i32(perm), dev(pw)]
    res = {}
    for tile in (64, 128):
        tl = np.array([(e, p) for e in range(E) for p in range(off[e], off[e + 1], tile)], np.int32)
        tb, nb = i32(tl), i32([len(tl)])
        g = group_args(W=bufs[0].ptr, w_gs=rows * cols, rows=rows, cols=cols, ldw=cols, n_group=E, x=bufs[1].ptr, ldx=cols, T=T, ldy=ldy, y_f32=y_f32, relu2=int(kind == "relu2"),
                       alpha=1.25, off=bufs[2].ptr, gather=bufs[3].ptr, gather_div=div, tiles=tb.ptr, n_tiles=nb.ptr, max_tiles=len(tl) + 3, glu=int(glu), glu_limit=5.0, glu_gain=1.5,
                       pair_w=bufs[4].ptr if kind == "pair" else None)
        print(rows, cols, kind, tile, flush=True)
        res[tile] = run(g, tile, n, ldy, y_f32)
    same(res[64][0], res[128][0], y_f32)
    if glu:
        return                                                                # (the small tiles' own tests hold them against float64)
    got = res[128][1]
    for e in range(E):
        s = slice(off[e], off[e + 1])
        want = 1.25 * (x[perm[s] // div].astype(np.float64) @ W[e].T.astype(np.float64))
        want = np.maximum(want, 0) ** 2 if kind == "relu2" else want
        if want.size:
            assert np.abs(got[s, :rows] - want).max() <= (1e-5 if y_f32 else 2.0 ** -7) * np.abs(want).max()


@pytest.mark.parametrize("groups,rows,cols,T", [(1, 512, 512, 2048), (3, 192, 256, 129), (2, 1024, 320, 40)])
def test_groups_without_a_list(groups, rows, cols, T):
    """Every group's own inputs, and more units than compute units."""
    rng = np.random.default_rng(T)
    W = rounded(rng.standard_normal((groups, rows, cols)) / np.sqrt(cols))
    x = rounded(rng.standard_normal((T, groups, cols)))
    wb, xb = store(W.reshape(-1, cols), pl.BF16), store(x.reshape(-1, cols), pl.BF16)
    ldy = groups * rows
    res = {}
    for tile in (64, 128):
        g = group_args(W=wb.ptr, w_gs=rows * cols, rows=rows, cols=cols, ldw=cols, n_group=groups, x=xb.ptr, x_gs=cols, ldx=groups * cols, T=T, y_gs=rows, ldy=ldy, alpha=1.0)
        print(groups, rows, cols, T, tile, flush=True)
        res[tile] = run(g, tile, T, ldy, 0)
    same(res[64][0], res[128][0], 0)
    want = np.einsum("tgc,grc->tgr", x.astype(np.float64), W.astype(np.float64)).reshape(T, ldy)
    assert np.abs(res[128][1] - want).max() <= 2.0 ** -7 * np.abs(want).max()


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("ff,cols,T", [(128, 256, 1), (384, 320, 64), (256, 512, 65), (640, 256, 129), (2176, 256, 300), (4352, 256, 3000)])
def test_sparse_ffn_of_a_chunk(ff, cols, T, gated):
    """Up, gate, mask and product in one kernel: h within fp16's rounding of float64 where the fp32 sums' own error leaves it (products of
    `cols` terms of fp16 values: 2^-11 of h and 1e-5 of the largest), exact zeros where the predictor says so, threshold and NaN included."""
    L, rng = pl.init(), np.random.default_rng(ff + T)
    up, gate, x = ((rng.standard_normal(s) / np.sqrt(s[1]) ** (s[0] != T)).astype(np.float16) for s in ((ff, cols), (ff, cols), (T, cols)))
    lg = rng.standard_normal((T, ff)).astype(np.float32)
    lg[0, :3] = [0.25, np.nan, -np.inf]
    b = [dev(a) for a in (up, gate, x, lg)]
    h = pl.DevBuf(2 * T * ff + 64)
    pl.check(L.pi_memset(h.ptr, 0xAB, h.nbytes))
    print(ff, cols, T, gated, flush=True)
    pl.check(L.pi_k_ffn_wide_f16(b[0].ptr, b[1].ptr if gated else None, ff, cols, b[2].ptr, T, b[3].ptr, 0.25, h.ptr, None))
    pl.sync()
    raw = h.download(np.float16)
    assert (raw[T * ff:].view(np.uint16) == 0xABAB).all()
    got = raw[:T * ff].reshape(T, ff).astype(np.float64)
    u, g = (x.astype(np.float64) @ w.T.astype(np.float64) for w in (up, gate))
    want = np.where(~(lg < 0.25), np.maximum(g, 0) * u if gated else np.maximum(u, 0), 0)
    assert (got[lg < 0.25] == 0).all()
    assert (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 1e-5 * np.abs(want).max() + 2.0 ** -25).all()


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("ff,rank,cols,T", [(128, 256, 256, 1), (384, 320, 256, 15), (128, 256, 320, 16), (256, 1024, 256, 17), (640, 256, 256, 64), (384, 256, 512, 65), (2176, 320, 256, 128),
                                            (640, 512, 256, 129), (1152, 256, 256, 301), (4352, 256, 256, 3000)])
def test_sparse_ffn_under_bits(ff, rank, cols, T, gated):
    """The predictor's second product leaves bits: factors are small whole numbers, whose sums fp32 holds exactly in any order, so that thresholds are met exactly
    (active) and missed by one; a token whose hidden vector has a NaN is active everywhere, infinite ones as their sums say.  The bits are
    float64's; h is bounded as above."""
    L, rng = pl.init(), np.random.default_rng(ff + T + rank)
    up, gate, x = ((rng.standard_normal(s) / np.sqrt(s[1]) ** (s[0] != T)).astype(np.float16) for s in ((ff, cols), (ff, cols), (T, cols)))
    fc2, hid = rng.integers(-3, 4, (ff, rank)).astype(np.float16), rng.integers(0, 3, (T, rank)).astype(np.float16)
    fc2[:, 5] = np.where(fc2[:, 5] == 0, 1, fc2[:, 5])
    if T > 2:
        hid[1, 7], hid[T - 1, 5] = np.nan, np.inf
    lg = (hid.astype(np.float64) @ fc2.astype(np.float64).T).astype(np.float32)
    thr = float(np.sort(lg[0])[ff // 2])
    active = ~(lg < thr)
    assert (lg[0] == thr).any() and active.any() and not active.all()
    b = [dev(a) for a in (fc2, hid, up, gate, x)]
    h, mask = pl.DevBuf(2 * T * ff + 64), pl.DevBuf((T + 15) // 16 * ff * 2 + 64)
    for d in (h, mask):
        pl.check(L.pi_memset(d.ptr, 0xAB, d.nbytes))
    print(ff, rank, cols, T, gated, flush=True)
    pl.check(L.pi_k_ffn_wide_predicted_f16(b[0].ptr, rank, b[1].ptr, b[2].ptr, b[3].ptr if gated else None, ff, cols, b[4].ptr, T, thr, mask.ptr, h.ptr, None))
    pl.sync()
    words, raw = mask.download(np.uint64), h.download(np.float16)
    assert (words[-8:] == 0xABABABABABABABAB).all() and (raw[T * ff:].view(np.uint16) == 0xABAB).all()
    bits = (words[:-8].reshape(-1, ff // 16, 4, 1) >> np.arange(64, dtype=np.uint64) & np.uint64(1)).reshape(-1, ff // 16, 4, 4, 16)      # [tile][neurons][r][l / 16][token]
    assert np.array_equal(bits.transpose(0, 4, 1, 3, 2).reshape(-1, ff)[:T] != 0, active)
    got = raw[:T * ff].reshape(T, ff).astype(np.float64)
    u, g = (x.astype(np.float64) @ w.T.astype(np.float64) for w in (up, gate))
    want = np.where(active, np.maximum(g, 0) * u if gated else np.maximum(u, 0), 0)
    assert (got[~active] == 0).all()
    assert (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 1e-5 * np.abs(want).max() + 2.0 ** -25).all()


def test_what_products_under_bits_refuse():
    L = pl.init()
    d = pl.DevBuf.zeros(1 << 20)
    call = lambda rank=256, ff=128, cols=256, fc2=d.ptr, mask=d.ptr, T=3: L.pi_k_ffn_wide_predicted_f16(fc2, rank, d.ptr, d.ptr, None, ff, cols, d.ptr, T, 0.0, mask, d.ptr, None)  # noqa: E731
    assert call(rank=128) != 0 and call(ff=64) != 0 and call(rank=300) != 0 and call(T=0) != 0 and call(fc2=d.ptr + 8) != 0 and call(mask=None) != 0 and call(mask=d.ptr + 8) != 0


def listed(counts, rows, cols, kind, y_f32, tile, tall):
    """One grouped product in tiles of `tile` tokens: what it wrote, as bits and as values, and float64 (None with a GLU)."""
    rng = np.random.default_rng(rows + cols)
    E, n, div = len(counts), sum(counts), 3
    T = (n + div - 1) // div
    W = rounded(rng.standard_normal((E, rows, cols), dtype=np.float32) / np.sqrt(cols))
    x = rounded(rng.standard_normal((T, cols), dtype=np.float32))
    perm = rng.permutation(T * div)[:n].astype(np.int32)
    pw = rng.random(T * div).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(counts)])
    glu = kind in ("glu", "pair")
    ldy = ((rows // 2 if glu else rows) + 7) // 8 * 8
    tl = np.array([(e, p) for e in range(E) for p in range(off[e], off[e + 1], tile)], np.int32)
    bufs = [store(W.reshape(-1, cols), pl.BF16), store(x, pl.BF16), i32(off), i32(perm), dev(pw), i32(tl), i32([len(tl)]), pl.DevBuf.zeros(4 * n * ldy + 64)]
    g = group_args(W=bufs[0].ptr, w_gs=rows * cols, rows=rows, cols=cols, ldw=cols, n_group=E, x=bufs[1].ptr, ldx=cols, T=T, ldy=ldy, y_f32=y_f32, relu2=int(kind == "relu2"),
                   alpha=1.25, off=bufs[2].ptr, gather=bufs[3].ptr, gather_div=div, tiles=bufs[5].ptr, n_tiles=bufs[6].ptr, max_tiles=len(tl) + 3, glu=int(glu), glu_limit=5.0, glu_gain=1.5,
                   pair_w=bufs[4].ptr if kind == "pair" else None, y=bufs[7].ptr)
    print(rows, cols, kind, tile, tall, flush=True)
    pl.check(pl.init().pi_k_group_gemm_tall(C.byref(g), None) if tall else pl.init().pi_k_group_gemm_tile(C.byref(g), tile, None))
    pl.sync()
    got = bufs[7].download(np.uint32 if y_f32 else np.uint16)
    assert not got[n * ldy:].any()
    want = None
    if not glu:
        want = np.concatenate([1.25 * (x[perm[off[e]:off[e + 1]] // div].astype(np.float64) @ W[e].T.astype(np.float64)) for e in range(E)])
        want = np.maximum(want, 0) ** 2 if kind == "relu2" else want
    return got[:n * ldy].reshape(n, ldy), fetch(bufs[7], pl.F32 if y_f32 else pl.BF16, (n, ldy))[:, :rows], want


COUNTS = [0, 1, 16, 63, 64, 65, 128, 129, 192, 193, 0, 255, 256, 257, 300, 40]


@pytest.mark.parametrize("rows,cols,kind,y_f32", [(72, 256, "plain", 0), (128, 320, "relu2", 0), (136, 256, "plain", 1), (192, 512, "glu", 0), (200, 256, "relu2", 0),
                                                  (270, 256, "plain", 0), (528, 384, "glu", 0), (400, 256, "pair", 0), (300, 256, "glu", 0)])
def test_tiles_of_256_tokens(rows, cols, kind, y_f32):
    """128 rows x 256 tokens: the sums of the small tiles, in their order."""
    small, _, _ = listed(COUNTS, rows, cols, kind, y_f32, 64, False)
    tall, got, want = listed(COUNTS, rows, cols, kind, y_f32, 256, True)
    same(small, tall, y_f32)
    if want is not None:
        assert np.abs(got - want).max() <= (1e-5 if y_f32 else 2.0 ** -7) * np.abs(want).max()


@pytest.mark.parametrize("rows,cols,tile", [(264, 2048, 128), (200, 4096, 256), (136, 2048, 256)])
def test_units_that_begin_at_other_columns(rows, cols, tile):
    """Rows a multiple of 4 KB apart: bf16 results of sums that begin at a column of the unit's own, within bf16's rounding of float64."""
    counts = [5, 70, 0, 129, 260, 33, 1, 100, 64, 7]
    _, got, want = listed(counts, rows, cols, "plain", 0, tile, tile == 256)
    assert np.linalg.norm(got - want) <= 2.0 ** -8 * np.linalg.norm(want) and np.abs(got - want).max() <= 2.0 ** -7 * np.abs(want).max()
    if tile == 128:
        _, got, want = listed(counts, rows, cols, "plain", 1, tile, False)
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("rows,cols,kind", [(264, 2048, "plain"), (520, 4096, "relu2"), (300, 4096, "plain"), (528, 2048, "glu"), (392, 4096, "pair"), (72, 4096, "plain")])
def test_one_order_of_sums_in_tiles_of_every_size(rows, cols, kind):
    """Rows a multiple of 4 KB apart, whose sums begin at columns of the group's and the row's own: the same in tiles of 64, 128 and 256 tokens, so that a token's outputs
    do not depend on the tile it falls into."""
    small, _, _ = listed(COUNTS, rows, cols, kind, 0, 64, False)
    for tile in (128, 256):
        other, _, _ = listed(COUNTS, rows, cols, kind, 0, tile, tile == 256)
        if kind in ("glu", "pair"):
            same(small, other, 0)
        else:
            assert np.array_equal(small, other), tile


@pytest.mark.parametrize("rows,cols,T", [(2304, 2048, 400), (1280, 5120, 300)])
def test_one_order_of_sums_without_a_list(rows, cols, T):
    """Small tiles, large ones, and large ones of other tokens beside these: the same bits."""
    rng = np.random.default_rng(T)
    wb, xb = store(rounded(rng.standard_normal((rows, cols)) / np.sqrt(cols)), pl.BF16), store(rounded(rng.standard_normal((T, cols))), pl.BF16)
    got = []
    for tile, n in ((64, T), (128, T), (128, T // 2)):
        g = group_args(W=wb.ptr, rows=rows, cols=cols, ldw=cols, n_group=1, x=xb.ptr, ldx=cols, T=n, ldy=rows, alpha=1.0)
        got.append(run(g, tile, n, rows, 0)[0])
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0][:T // 2], got[2])


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("ff,cols", [(2304, 4096), (4352, 8192)])
def test_a_chunks_neurons_do_not_depend_on_its_length(ff, cols, gated):
    """The sparse FFN's large tiles: the first tokens of a chunk have the same bits whatever follows them."""
    L, rng = pl.init(), np.random.default_rng(ff)
    T = 300
    up, gate, x = (dev((rng.standard_normal(s, dtype=np.float32) / np.sqrt(s[1]) ** (s[0] != T)).astype(np.float16)) for s in ((ff, cols), (ff, cols), (T, cols)))
    lg = dev(rng.standard_normal((T, ff)).astype(np.float32))
    got = []
    for n in (T, 129, 70):
        h = pl.DevBuf.zeros(2 * T * ff)
        print(ff, cols, n, gated, flush=True)
        pl.check(L.pi_k_ffn_wide_f16(up.ptr, gate.ptr if gated else None, ff, cols, x.ptr, n, lg.ptr, 0.25, h.ptr, None))
        pl.sync()
        got.append(h.download(np.uint16)[:n * ff].reshape(n, ff))
    for g in got[1:]:
        assert np.array_equal(got[0][:len(g)], g)


def test_what_tiles_of_256_tokens_do_not_cover_is_refused():
    L, b = pl.init(), pl.DevBuf(1 << 16)
    p = lambda **kw: C.byref(group_args(**dict(dict(W=b.ptr, rows=128, cols=256, ldw=256, n_group=1, x=b.ptr, ldx=256, T=8, y=b.ptr, ldy=128, alpha=1.0, off=b.ptr, tiles=b.ptr, n_tiles=b.ptr, max_tiles=1), **kw)))  # noqa: E731
    for bad in (dict(off=None), dict(rows=64), dict(cols=192), dict(cols=250), dict(max_tiles=0)):
        assert L.pi_k_group_gemm_tall(p(**bad), None) != 0, bad
    assert L.pi_k_group_gemm_tile(p(), 256, None) != 0
