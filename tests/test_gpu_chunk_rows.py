"""Attention of long prompt chunks, 64 or 128 tokens of a head per workgroup (attn_chunk_rows_kernel): against float64 on the rounded
operands, at the edges of its row and cell tiles, and with values that are no numbers in cells that a token does not see."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rotated(x, pos, mode, hd):
    """x [T, heads, hd]; the angles in float32, advanced by repeated products as the kernels form them."""
    scale = np.float32(np.float32(10000.0) ** np.float32(-2.0 / hd))
    th = np.empty((len(pos), hd // 2), np.float32)
    th[:, 0] = pos
    for i in range(1, hd // 2):
        th[:, i] = th[:, i - 1] * scale
    c, s = np.cos(th)[:, None].astype(np.float64), np.sin(th)[:, None].astype(np.float64)
    a, b = (slice(0, hd // 2), slice(hd // 2, hd)) if mode == 2 else (slice(0, hd, 2), slice(1, hd, 2))
    y = np.empty(x.shape)
    y[..., a], y[..., b] = x[..., a] * c - x[..., b] * s, x[..., a] * s + x[..., b] * c
    return y


def run(hd, nh, nkv, mode, past, T, n_ctx, spoil=None):
    from powerinfer_amd import lib as pl
    L = pl.init()
    rng = np.random.default_rng(hd + nh + past + T)
    gqa, d = nkv * hd, nh * hd
    kc = rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16)
    vc = rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16)
    kc[:, past + T:], vc[:, past + T:] = np.nan, np.nan                     # cells never written
    qkv = rng.standard_normal((T, d + 2 * gqa)).astype(np.float32)
    if spoil is not None:
        qkv[spoil, d + gqa:] = np.inf
    pos = np.arange(past, past + T, dtype=np.int32)
    dq, dpos, dk, dv = pl.DevBuf(host=qkv), pl.DevBuf(host=pos), pl.DevBuf(host=kc), pl.DevBuf(host=vc)
    rot, out, out16 = pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 2)
    pl.check(L.pi_memset(out.ptr, 0xFF, out.nbytes), "memset")
    theta = float(np.float32(10000.0) ** np.float32(-2.0 / hd))
    print("rows", hd, nh, nkv, mode, past, T, flush=True)
    pl.check(L.pi_k_attn_chunk_rows(dq.ptr, d + 2 * gqa, T, nh, nkv, hd, mode, theta, 1.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, out.ptr, d, out16.ptr, None), "attn_chunk_rows")
    pl.sync()
    got = out.download(np.float32).reshape(T, nh, hd)
    with np.errstate(invalid="ignore", over="ignore"):
        assert np.array_equal(out16.download(np.float16).reshape(T, nh, hd), got.astype(np.float16), equal_nan=True)
    k, v = dk.download(np.float16).reshape(nkv, n_ctx, hd).astype(np.float64), dv.download(np.float16).reshape(nkv, n_ctx, hd).astype(np.float64)
    want_k = rotated(qkv[:, d:d + gqa].reshape(T, nkv, hd), pos, mode, hd).transpose(1, 0, 2)
    assert np.abs(k[:, past:past + T] - want_k).max() < 4e-3 * np.abs(want_k).max()               # rounded to fp16
    assert np.array_equal(v[:, past:past + T], qkv[:, d + gqa:].reshape(T, nkv, hd).transpose(1, 0, 2).astype(np.float16).astype(np.float64), equal_nan=True)
    q = rotated(qkv[:, :d].reshape(T, nh, hd), pos, mode, hd).astype(np.float16).astype(np.float64)
    heads = range(nh) if nh <= 8 else sorted(set(rng.integers(0, nh, 6)) | {0, nh - 1})
    seen = np.arange(past + T)[None] <= pos[:, None]
    want = {}
    for a in heads:
        g = a * nkv // nh
        s = np.where(seen, q[:, a] @ k[g, :past + T].T / np.sqrt(hd), -np.inf)
        e = np.exp(s - s.max(1, keepdims=True))
        e /= e.sum(1, keepdims=True)
        want[a] = e @ (v[g, :past + T] if spoil is None else np.where(np.isfinite(v[g, :past + T]), v[g, :past + T], 0))
    return got, want


# fp16(s - max) is off by up to 2^-10 for |s - max| in [2, 4) and the weight by as much of itself, 6e-4 in the root mean square of a row
@pytest.mark.parametrize("hd,nh,nkv,mode,past,T,n_ctx", [
    (128, 4, 4, 0, 0, 1, 64), (128, 4, 4, 0, 0, 63, 64), (128, 4, 4, 0, 1, 64, 96), (128, 4, 2, 0, 63, 65, 160), (64, 8, 2, 2, 0, 127, 160), (64, 4, 4, 0, 64, 128, 192),
    (64, 8, 1, 2, 5, 129, 160), (128, 2, 2, 2, 1900, 90, 2400), (128, 2, 1, 0, 0, 700, 736), (64, 256, 8, 2, 30, 129, 160), (128, 256, 8, 0, 3, 190, 224)])
def test_rows_match_float64(hd, nh, nkv, mode, past, T, n_ctx):
    got, want = run(hd, nh, nkv, mode, past, T, n_ctx)
    for a, w in want.items():
        err = np.linalg.norm(got[:, a] - w) / np.linalg.norm(w)
        assert err < 2e-3, (a, err)


def exact_weights(T, past, seed, whole, n_ctx):
    """Scores, cells and queries that every step up to the weights forms without rounding but the CPU path's own: (qkv, K, V, what comes out bit
    for bit).  Scores are multiples of 1/128, the values of cell c a one in column c % 64, so that a column is the exact sum of its
    cells' weights.  whole: the weights are not divided by their sum before they meet the values."""
    hd = 64
    rng = np.random.default_rng(seed)
    q, k = np.zeros((T, hd), np.float32), np.zeros((past + T, hd), np.float32)
    q[:, 0], q[:, 1] = rng.integers(1, 4, T) / 4, 1
    k[:, 0], k[:, 1] = rng.integers(-60, 1, past + T), rng.integers(-8, 9, past + T) * 0.25          # s / 8: -5.6 q .. 0.3
    k[rng.integers(0, past + T, 3 + (past + T) // 40), 0] = rng.integers(20, 90)
    v = np.zeros((past + T, hd), np.float16)
    v[np.arange(past + T), np.arange(past + T) % hd] = 1
    s = (q.astype(np.float64) @ k.T.astype(np.float64)).astype(np.float32) * np.float32(0.125)
    seen = np.arange(past + T)[None] <= (past + np.arange(T))[:, None]
    x = np.where(seen, s - np.where(seen, s, -np.inf).max(1, keepdims=True), -np.inf)
    x = x if whole else x.astype(np.float16)
    ex = np.exp(x.astype(np.float64))
    e = ex.astype(np.float16)
    vals = np.unique(ex[seen])                                            # no exponential lies within two units of float32 of where fp16 rounds the other way
    for d in (-2, 2):
        assert np.array_equal((vals * (1 + d * 2.0 ** -23)).astype(np.float16), vals.astype(np.float16))
    total = e.astype(np.float64).sum(1, keepdims=True)
    w = e.astype(np.float64) if whole else (e.astype(np.float32) * (1.0 / total).astype(np.float32)).astype(np.float16).astype(np.float64)
    out = w @ v.astype(np.float64)
    if whole:
        out = (out.astype(np.float32) / total.astype(np.float32)).astype(np.float64)
    qkv = np.concatenate([q, k[past:], v[past:].astype(np.float32)], 1)
    kc, vc = np.full((n_ctx, hd), np.nan, np.float16), np.full((n_ctx, hd), np.nan, np.float16)
    kc[:past], vc[:past] = k[:past], v[:past]
    return qkv, kc, vc, out


def rows_of(qkv, kc, vc, T, past, n_ctx):
    from powerinfer_amd import lib as pl
    L = pl.init()
    dq, dk, dv, dpos = pl.DevBuf(host=qkv), pl.DevBuf(host=kc), pl.DevBuf(host=vc), pl.DevBuf(host=np.arange(past, past + T, dtype=np.int32))
    rot, out = pl.DevBuf(T * 64 * 4), pl.DevBuf(T * 64 * 4)
    pl.check(L.pi_k_attn_chunk_rows(dq.ptr, 192, T, 1, 1, 64, 0, 1.0, 0.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, out.ptr, 64, None, None), "attn_chunk_rows")
    pl.sync()
    return out.download(np.float32).reshape(T, 64)


@pytest.mark.parametrize("T,past", [(700, 0), (130, 1500), (40, 300), (1900, 148)])
def test_weights_are_those_of_a_sum_in_double_bit_for_bit(T, past):
    """The soft-max's sum holds every bit of its weights, large and subnormal ones in one tile: 1 / sum, and with it the rounding of each
    weight to fp16, are the CPU path's."""
    wrong, n_ctx = 0, past + T + 8
    for seed in range(4):
        qkv, kc, vc, want = exact_weights(T, past, 100 * seed + T, False, n_ctx)
        wrong += int((rows_of(qkv, kc, vc, T, past, n_ctx) != want).any(1).sum())
    assert wrong == 0, f"{wrong} of {4 * T} rows"


@pytest.mark.parametrize("T,past", [(70, 2600), (700, 2400), (2048, 500)])
def test_weights_of_a_large_cache_are_divided_once_in_float32(T, past):
    """Caches beyond what decoding holds in one workgroup: as in pi_k_attn_chunk_long, which took these chunks, a weight meets its value as fp16(exp)
    and the fp32 result is divided.  Sums of 40 such products are within 40 units of 2^-24 of the whole, the division within two."""
    from powerinfer_amd import lib as pl
    n_ctx = 14000
    assert not pl.init().pi_k_attn_chunk_supported(64, n_ctx, past + T)
    qkv, kc, vc, want = exact_weights(T, past, T, True, n_ctx)
    got = rows_of(qkv, kc, vc, T, past, n_ctx)
    err = np.abs(got - want).max(1) / np.abs(want).max(1)
    assert err.max() < 42 * 2.0 ** -24, err.max()


@pytest.mark.parametrize("hd,T,past", [(128, 40, 2500), (64, 130, 2600)])
def test_no_further_from_float64_than_the_kernel_that_splits_cells(hd, T, past):
    """Against pi_k_attn_chunk_long on one cache, which rounds fp16(s - max of the part) and fp16(exp); here only the latter."""
    from powerinfer_amd import lib as pl
    L = pl.init()
    n_ctx, nh, parts = 14000, 4, 4
    rng = np.random.default_rng(T)
    d = nh * hd
    kc, vc = rng.standard_normal((nh, n_ctx, hd)).astype(np.float16), rng.standard_normal((nh, n_ctx, hd)).astype(np.float16)
    qkv = rng.standard_normal((T, 3 * d)).astype(np.float32)
    pos = np.arange(past, past + T, dtype=np.int32)
    dq, dpos, dk, dv = pl.DevBuf(host=qkv), pl.DevBuf(host=pos), pl.DevBuf(host=kc), pl.DevBuf(host=vc)
    rot, out, scr = pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 4), pl.DevBuf(int(L.pi_k_attn_split_scratch_floats(T, nh, hd, parts)) * 4)
    theta, got = float(np.float32(10000.0) ** np.float32(-2.0 / hd)), []
    for rows in (True, False):
        if rows:
            rc = L.pi_k_attn_chunk_rows(dq.ptr, 3 * d, T, nh, nh, hd, 0, theta, 1.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, out.ptr, d, None, None)
        else:
            rc = L.pi_k_attn_chunk_long(dq.ptr, 3 * d, T, nh, nh, hd, 0, theta, 1.0, dpos.ptr, n_ctx, parts, scr.ptr, rot.ptr, dk.ptr, dv.ptr, out.ptr, None, None)
        pl.check(rc, "attention")
        pl.sync()
        got.append(out.download(np.float32).reshape(T, nh, hd).astype(np.float64))
    k, v = dk.download(np.float16).reshape(nh, n_ctx, hd).astype(np.float64), dv.download(np.float16).reshape(nh, n_ctx, hd).astype(np.float64)
    q = rot.download(np.float32).reshape(T, nh, hd).astype(np.float16).astype(np.float64)
    want = np.empty((T, nh, hd))
    for a in range(nh):
        s = np.where(np.arange(past + T)[None] <= pos[:, None], q[:, a] @ k[a, :past + T].T / np.sqrt(hd), -np.inf)
        e = np.exp(s - s.max(1, keepdims=True))
        want[:, a] = e / e.sum(1, keepdims=True) @ v[a, :past + T]
    errs = [np.linalg.norm(g - want) / np.linalg.norm(want) for g in got]
    assert errs[0] <= errs[1], errs


def test_what_it_does_not_cover_is_refused():
    from powerinfer_amd import lib as pl
    L, b = pl.init(), pl.DevBuf(1 << 16)
    call = lambda hd, stride: L.pi_k_attn_chunk_rows(b.ptr, 3 * hd, 2, 1, 1, hd, 0, 0.9, 1.0, b.ptr, 8, 4, b.ptr, b.ptr, b.ptr, b.ptr, stride, None, None)  # noqa: E731
    assert call(32, 32) != 0 and call(64, 66) != 0
    assert not L.pi_k_attn_chunk_rows_supported(32, 64, 64) and not L.pi_k_attn_chunk_rows_supported(64, 16, 64) and L.pi_k_attn_chunk_rows_supported(64, 17, 64)


@pytest.mark.parametrize("hd,T,spoil", [(128, 70, 40), (64, 150, 149), (128, 40, 0)])
def test_a_value_that_is_no_number_reaches_the_tokens_that_see_it_only(hd, T, spoil):
    got, want = run(hd, 2, 2, 0, 10, T, 192, spoil=spoil)
    for a, w in want.items():
        assert np.isfinite(got[:spoil, a]).all() and not np.isfinite(got[spoil:, a]).any()
        if spoil:
            assert np.linalg.norm(got[:spoil, a] - w[:spoil]) / np.linalg.norm(w[:spoil]) < 2e-3
