"""What a long pass does a row at a time: the router's product in parts with the choice behind it, norms of rows into one operand or two, normed embeddings, at edges of
the tiles and of what the registers hold."""
import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_latent_ops import TYPES, dev, fetch, i32, store, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [17, 64, 65, 130])
@pytest.mark.parametrize("E,top,groups,keep", [(64, 6, 8, 4), (64, 6, 1, 1), (1, 1, 1, 1), (17, 5, 1, 1), (128, 8, 4, 2), (6, 2, 3, 2)])
@pytest.mark.parametrize("cols,biased", [(512, True), (4096, True), (1536, False)])
def test_choice_behind_the_product(T, E, top, groups, keep, cols, biased):
    if not biased and groups > 1:
        return
    L, rng = pl.init(), np.random.default_rng(T + E + cols)
    Wb, xb = store(rng.standard_normal((E, cols)), pl.BF16), store(rng.standard_normal((T, cols)) * cols ** -0.5, pl.BF16)
    bias = rng.standard_normal(E).astype(np.float32) * 0.1
    bb = dev(bias) if biased else None
    n = L.pi_k_router_parts(T, E, cols)
    assert n == cols // 512
    parts, ids, wts = dev(np.full(n * T * E, np.nan, np.float32)), pl.DevBuf.zeros(4 * T * top), pl.DevBuf.zeros(4 * T * top)
    print(T, E, cols, groups, biased, flush=True)
    pl.check(L.pi_k_route_long(Wb.ptr, E, cols, xb.ptr, T, parts.ptr, top, groups, keep, bb.ptr if biased else None, ids.ptr, wts.ptr, None))
    pl.sync()
    W, x = fetch(Wb, pl.BF16, (E, cols)).astype(np.float64), fetch(xb, pl.BF16, (T, cols)).astype(np.float64)
    z, off = x @ W.T, np.abs(x) @ np.abs(W).T * cols * 2.0 ** -24
    got = parts.download(np.float32).reshape(n, T, E).sum(0)
    assert (np.abs(got - z) <= off).all()
    # the operator without the product, on the sums: the same choice and weights up to the last place of a sum
    s = dev(got)
    ids2, wts2 = pl.DevBuf.zeros(4 * T * top), pl.DevBuf.zeros(4 * T * top)
    if biased:
        pl.check(L.pi_k_route(s.ptr, T, E, top, groups, keep, bb.ptr, ids2.ptr, wts2.ptr, None))
    else:
        pl.check(L.pi_k_route_scores(s.ptr, T, E, top, ids2.ptr, wts2.ptr, None))
    pl.sync()
    a, b = ids.download(np.int32).reshape(T, top), ids2.download(np.int32).reshape(T, top)
    w1, w2 = wts.download(np.float32).reshape(T, top), wts2.download(np.float32).reshape(T, top)
    same = (a == b).all(1)                                            # (sums of the parts in another order: a tie within a last place may fall the other way)
    assert same.mean() > 0.95 and np.abs(w1[same] - w2[same]).max() < 1e-5


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("T,cols,two,ol,some", [(1, 4096, True, 1, False), (5, 4, False, 0, False), (3, 1024, True, 0, True), (16, 1028, True, 0, False), (2, 4100, True, 0, False), (33, 2052, False, 0, True), (4, 99, True, 0, False), (17, 4, True, 0, False), (40, 4096, True, 0, True), (18, 1028, False, 0, False), (19, 4100, True, 0, False)])
def test_norms_into_operands(t, T, cols, two, ol, some):
    if ol and t == pl.F32:
        return
    L, rng = pl.init(), np.random.default_rng(T + cols)
    ld, n = (cols + 63) // 64 * 64, T + 3
    x, wa, wb = rng.standard_normal((n, cols)).astype(np.float32), rng.random(cols).astype(np.float32), rng.random(cols).astype(np.float32)
    rows = rng.permutation(n)[:T] if some else np.arange(T)
    xb, ab, bb, rb = dev(x), dev(wa), dev(wb), i32(rows.astype(np.int32))
    a, b = pl.DevBuf.zeros(4 * max(T, 16) * ld), pl.DevBuf.zeros(4 * max(T, 16) * ld)
    print(t, T, cols, two, ol, some, flush=True)
    pl.check(L.pi_k_norm_pair(t, xb.ptr, rb.ptr if some else None, T, cols, 1e-5, ab.ptr, a.ptr, bb.ptr if two else None, b.ptr if two else None, ld, ol, None))
    pl.sync()
    v = x[rows].astype(np.float64)
    v = v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5)
    for buf, w in ((a, wa), (b, wb))[:1 + two]:
        got = fetch(buf, t, (ld // 8, 16, 8)).transpose(1, 0, 2).reshape(16, ld)[:T, :cols] if ol else fetch(buf, t, (T, ld))[:, :cols]
        assert np.abs(got - v * w).max() <= tol(t, 1) * np.abs(v * w).max()


@pytest.mark.parametrize("cols", [8, 4096, 2056, 8192, 8200, 99])
def test_normed_embeddings(cols):
    L, rng = pl.init(), np.random.default_rng(cols)
    table, w, toks = rng.standard_normal((11, cols)), rng.random(cols).astype(np.float32), np.array([3, 10, 0, 3, 7], np.int32)
    tb, wb, kb, x = store(table, pl.BF16), dev(w), i32(toks), pl.DevBuf.zeros(4 * 5 * cols)
    print(cols, flush=True)
    pl.check(L.pi_k_embed_norm(tb.ptr, cols, kb.ptr, 5, wb.ptr, 1e-5, x.ptr, None))
    pl.sync()
    v = fetch(tb, pl.BF16, (11, cols)).astype(np.float64)[toks]
    want = v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5) * w
    assert np.abs(x.download(np.float32).reshape(5, cols) - want).max() < 1e-6 * np.abs(want).max()
