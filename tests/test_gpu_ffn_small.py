"""The sparse FFN of a small F16 layer, predictor included, in one launch and a reduction: against float64, over the smallest and largest of its range,
with and without gate and norm, with no, some and every neuron active.  Rows of inactive neurons hold NaN: none of them may be read into the result."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_short_rows import normed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ff,r,cols", [(32, 64, 512), (96, 128, 512), (4096, 256, 512), (4128, 64, 1024), (1024, 128, 1024), (8192, 64, 512)])
@pytest.mark.parametrize("kind,gate,active", [(0, False, "some"), (1, True, "some"), (2, False, "all"), (1, True, "none"), (2, True, "some")])
def test_small_ffn_in_one_launch(ff, r, cols, kind, gate, active):
    L, rng = pl.init(), np.random.default_rng(ff + r + cols + kind)
    half = lambda *s: (rng.standard_normal(s) * s[-1] ** -0.5).astype(np.float16)
    fc1, fc2, up, gt, down = half(r, cols), half(ff, r), half(ff, cols), half(ff, cols), half(ff, cols)
    x, w, b, a1, a2 = (rng.standard_normal(cols).astype(np.float32) + np.float32(0.5) for _ in range(5))
    x16 = x.astype(np.float16).astype(np.float64)
    hid = np.maximum(fc1.astype(np.float64) @ x16, 0)
    lg = fc2.astype(np.float64) @ hid.astype(np.float16).astype(np.float64)
    # a threshold in the widest gap between the logits around a tenth of them
    top = np.sort(lg)[::-1][max(1, ff // 16):max(3, ff // 8)]
    cut = int(np.argmax(top[:-1] - top[1:]))
    thr = {"some": (top[cut] + top[cut + 1]) / 2, "all": -np.inf, "none": np.inf}[active]
    on = lg >= thr
    # hidden units: sums of cols products in fp32, then one fp16 rounding that may fall the other way; no logit may lie closer to the line than that
    # (the few that do are moved off it: their fc2 row becomes one that the hidden units cannot raise)
    off = np.abs(fc2.astype(np.float64)) @ (hid * 2.0 ** -10 + np.abs(fc1.astype(np.float64)) @ np.abs(x16) * cols * 2.0 ** -24)
    if active == "some":
        near = np.abs(lg - thr) <= off
        fc2[near] = -np.abs(fc2[near])
        on &= ~near
    for m in (up, gt, down):
        m[~on] = np.nan
    bufs = [pl.DevBuf(host=v) for v in (fc1, fc2, up, gt, down, x, w, b, a1, a2)]
    d1, d2, du, dg, dd, dx, dw, db, da1, da2 = (v.ptr for v in bufs)
    out, n = pl.DevBuf(host=np.full(cols, np.nan, np.float32)), pl.DevBuf(host=np.full(1, -1, np.int32))
    ws = L.pi_workspace_create(ff, cols)
    nrm = pl.Norm(kind, 1e-5, dw if kind else None, db if kind == 2 else None)
    print(ff, r, cols, kind, gate, active, flush=True)
    assert L.pi_k_sparse_ffn_small_supported(ff, r, cols)
    pl.check(L.pi_k_sparse_ffn_small(d1, d2, ff, r, float(thr), du, dg if gate else None, dd, cols, dx, C.byref(nrm), pl.EPI_ADD2, da1, da2, out.ptr, n.ptr, ws, None), "small")
    got = out.download(np.float32)
    L.pi_workspace_destroy(ws)
    assert n.download(np.int32)[0] == on.sum()
    # products of the fp16-rounded input (2^-11 of each, a few 2^-24 from the norm), h rounded once more, all sums in fp32
    xn = normed(x, kind, w, b) if kind else x16
    U, G, D = (m[on].astype(np.float64) for m in (up, gt, down))
    rel = (2.0 ** -11 + 2.0 ** -20 if kind else 0) + cols * 2.0 ** -24
    u, eu = U @ xn, np.abs(U) @ np.abs(xn) * rel
    g, eg = G @ xn, np.abs(G) @ np.abs(xn) * rel
    h = np.maximum(g, 0) * u if gate else np.maximum(u, 0)
    eh = (eg * np.abs(u) + np.maximum(g, 0) * eu + eg * eu if gate else eu)
    eh = eh + (np.abs(h) + eh) * 2.0 ** -11 + 2.0 ** -25
    want = h @ D + a1 + a2
    bound = eh @ np.abs(D) + (np.abs(h) @ np.abs(D)) * (on.sum() + 8) * 2.0 ** -24 + (np.abs(want) + np.abs(a1) + np.abs(a2)) * 2.0 ** -22
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("cols,gate", [(512, True), (1024, False)])
def test_active_neurons_of_value_zero(cols, gate):
    """Neurons that the predictor calls active and whose value is zero, or rounds to zero in fp16, add nothing, whatever their rows of the down projection hold."""
    L, rng = pl.init(), np.random.default_rng(cols)
    ff, r = 256, 64
    half = lambda *s: (rng.standard_normal(s) * s[-1] ** -0.5).astype(np.float16)
    fc1, fc2, up, gt, down = half(r, cols), half(ff, r), half(ff, cols), half(ff, cols), half(ff, cols)
    x = np.abs(rng.standard_normal(cols)).astype(np.float32)
    zero, tiny, bad = np.arange(0, ff, 3), np.arange(1, ff, 9), np.float16(np.inf)
    (gt if gate else up)[zero] = -np.abs((gt if gate else up)[zero])          # negative products of positive inputs
    up[tiny] = 0
    if gate:
        gt[tiny] = np.abs(gt[tiny])
        up[tiny, 0], x[0] = np.float16(6e-8), np.float32(2.0 ** -14)          # a product far below fp16's smallest value
    down[zero], down[tiny, ::2], down[tiny, 1::2] = bad, -bad, np.nan
    bufs = [pl.DevBuf(host=v) for v in (fc1, fc2, up, gt, down, x)]
    d1, d2, du, dg, dd, dx = (v.ptr for v in bufs)
    out, n = pl.DevBuf(host=np.full(cols, np.nan, np.float32)), pl.DevBuf(host=np.full(1, -1, np.int32))
    ws, nrm = L.pi_workspace_create(ff, cols), pl.Norm(0, 1e-5, None, None)
    pl.check(L.pi_k_sparse_ffn_small(d1, d2, ff, r, float("-inf"), du, dg if gate else None, dd, cols, dx, C.byref(nrm), 0, None, None, out.ptr, n.ptr, ws, None), "small")
    got = out.download(np.float32)
    L.pi_workspace_destroy(ws)
    assert n.download(np.int32)[0] == ff
    keep = np.ones(ff, bool)
    keep[zero] = keep[tiny] = False
    x64 = x.astype(np.float16).astype(np.float64)
    U, G, D = (m[keep].astype(np.float64) for m in (up, gt, down))
    h = np.maximum(G @ x64, 0) * (U @ x64) if gate else np.maximum(U @ x64, 0)
    eh = (np.abs(G) @ x64) * (np.abs(U) @ x64) * cols * 2.0 ** -22 if gate else (np.abs(U) @ x64) * cols * 2.0 ** -24
    bound = (eh + np.abs(h) * 2.0 ** -11 + 2.0 ** -25) @ np.abs(D) + (np.abs(h) @ np.abs(D)) * (ff + 8) * 2.0 ** -24
    assert (np.abs(got - h @ D) <= bound).all()


def test_refusals():
    L = pl.init()
    for ff, r, cols in ((48, 128, 512), (0, 128, 512), (4096, 512, 512), (4096, 256, 1024), (4096, 128, 768), (4096, 96, 512)):
        assert not L.pi_k_sparse_ffn_small_supported(ff, r, cols)
