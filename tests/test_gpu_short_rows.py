"""F16 mat-vec and predictor products at shapes without a kernel of their own: rows that end inside the first columns requested ahead of the
input, exactly on them and behind them, waves and lanes past the matrix, inputs held in registers (at most 1024 values) and longer ones."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


def normed(x, kind, w, b, eps=1e-5):
    v = x.astype(np.float64)
    if kind == 2:
        v = v - v.mean()
    if kind:
        v = v / np.sqrt((v * v).mean() + eps)
        v = v * w + (b if kind == 2 else 0)
    return v


@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 504), (9, 520), (3, 1024), (6, 1032), (7, 2040), (2, 2056), (4, 2568), (8203, 24)])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_gemv_f16_any_shape(rows, cols, kind):
    L, rng = pl.init(), np.random.default_rng(rows + cols + kind)
    W = rng.standard_normal((rows, cols)).astype(np.float16)
    x = rng.standard_normal(cols).astype(np.float32) + np.float32(0.5)
    w, b, add = (rng.standard_normal(n).astype(np.float32) for n in (cols, cols, rows))
    dW, dx, dw, db, da, dy = (pl.DevBuf(host=a) for a in (W, x, w, b, add, np.zeros(rows, np.float32)))
    nrm = pl.Norm(kind, 1e-5, dw.ptr, db.ptr if kind == 2 else None)
    print(rows, cols, kind, flush=True)
    pl.check(L.pi_k_gemv(pl.F16, dW.ptr, rows, cols, dx.ptr, C.byref(nrm) if kind else None, pl.EPI_ADD, da.ptr, None, dy.ptr, None), "gemv")
    y, xn = dy.download(np.float32), normed(x, kind, w, b)
    want = W.astype(np.float64) @ (xn if kind else x.astype(np.float16).astype(np.float64)) + add
    # the input rounded to fp16 (2^-11 of each product; of the norm, computed in fp32, a few 2^-24 more), sums of cols products in fp32
    bound = np.abs(W.astype(np.float64)) @ np.abs(xn) * ((2.0 ** -11 + 2.0 ** -21 if kind else 0) + cols * 2.0 ** -24) + np.abs(want) * 2.0 ** -23 + 1e-7
    assert (np.abs(y - want) <= bound).all()


@pytest.mark.parametrize("ff,r", [(1, 8), (33, 128), (31, 504), (40, 520), (70, 1032), (64, 1016), (100, 2048)])
def test_predictor_any_rank(ff, r):
    L, rng = pl.init(), np.random.default_rng(ff + r)
    W, hid = rng.standard_normal((ff, r)).astype(np.float16), rng.standard_normal(r).astype(np.float32)
    W[ff // 2, r - 1] = np.inf                                       # stays in its row
    dW, dh, lg, rows, n = (pl.DevBuf(host=a) for a in (W, hid, np.zeros(ff, np.float32), np.zeros(ff, np.int32), np.zeros(1, np.int32)))
    ws = L.pi_workspace_create(ff, 64)
    print(ff, r, flush=True)
    pl.check(L.pi_k_predictor_fc2(dW.ptr, ff, r, dh.ptr, 0.25, None, 0, lg.ptr, rows.ptr, n.ptr, None, ws, None), "fc2")
    got, h16 = lg.download(np.float32), hid.astype(np.float16).astype(np.float64)
    active = rows.download(np.int32)[:n.download(np.int32)[0]]
    L.pi_workspace_destroy(ws)
    fin = np.arange(ff) != ff // 2
    want, mag = W[fin].astype(np.float64) @ h16, np.abs(W[fin].astype(np.float64)) @ np.abs(h16)
    assert (np.abs(got[fin] - want) <= mag * r * 2.0 ** -24).all() and np.isinf(got[ff // 2])
    assert np.array_equal(active, np.flatnonzero(got >= 0.25))
