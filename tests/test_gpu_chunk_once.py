"""Attention of F16 prompt chunks in one pass over the keys (attn_chunk_rows_once_kernel): its queries and cells are those of the three-pass kernel
bit for bit, its result is held against float64 on them, at the edges of row and cell tiles, with scores that keep raising a row's
base, and with values that are no numbers in cells that a token does not see."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(hd, nh, nkv, mode, past, T, n_ctx, grow=0.0, spoil=None):
    from powerinfer_amd import lib as pl
    L = pl.init()
    rng = np.random.default_rng(hd + nh + past + T)
    gqa, d = nkv * hd, nh * hd
    kc = rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16)
    vc = rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16)
    kc[:, past + T:], vc[:, past + T:] = np.nan, np.nan                     # cells never written
    qkv = rng.standard_normal((T, d + 2 * gqa)).astype(np.float32)
    theta = float(np.float32(10000.0) ** np.float32(-2.0 / hd))
    if grow:                                                                # positive queries and keys that grow with their cell (nothing turned: the angles are 0)
        theta, scale = 0.0, np.linspace(0, grow, past + T)
        kc[:, :past + T] = (np.abs(kc[:, :past + T]) * scale[None, :, None]).astype(np.float16)
        qkv[:, :d], qkv[:, d:d + gqa] = np.abs(qkv[:, :d]), np.abs(qkv[:, d:d + gqa]) * scale[past:, None]
    if spoil is not None:
        qkv[spoil, d + gqa:] = np.inf
    pos = np.arange(past, past + T, dtype=np.int32)
    dq, dpos = pl.DevBuf(host=qkv), pl.DevBuf(host=pos)
    rot, out, q16, out16 = pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 2), pl.DevBuf(T * d * 2)
    caches = []
    for once in (False, True):
        dk, dv = pl.DevBuf(host=kc), pl.DevBuf(host=vc)
        print("once" if once else "rows", hd, nh, nkv, mode, past, T, flush=True)
        if once:
            pl.check(L.pi_k_attn_chunk_once(dq.ptr, d + 2 * gqa, T, nh, nkv, hd, mode, theta, 0.0 if grow else 1.0, dpos.ptr, n_ctx, past + T, q16.ptr, dk.ptr, dv.ptr, out.ptr, d, out16.ptr, None), "attn_chunk_once")
        else:
            pl.check(L.pi_k_attn_chunk_rows(dq.ptr, d + 2 * gqa, T, nh, nkv, hd, mode, theta, 0.0 if grow else 1.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, out.ptr, d, None, None), "attn_chunk_rows")
        pl.sync()
        caches.append((dk.download(np.float16), dv.download(np.float16)))
    for a, b in zip(*caches):
        assert np.array_equal(a, b, equal_nan=True)
    q = q16.download(np.float16)
    assert np.array_equal(q, rot.download(np.float32).astype(np.float16))
    got = out.download(np.float32).reshape(T, nh, hd)
    with np.errstate(invalid="ignore", over="ignore"):
        assert np.array_equal(out16.download(np.float16).reshape(T, nh, hd), got.astype(np.float16), equal_nan=True)
    k, v = (c.reshape(nkv, n_ctx, hd)[:, :past + T].astype(np.float64) for c in caches[1])
    q = q.reshape(T, nh, hd).astype(np.float64)
    seen = np.arange(past + T)[None] <= pos[:, None]
    want = {}
    for a in range(nh) if nh <= 8 else sorted(set(rng.integers(0, nh, 6)) | {0, nh - 1}):
        g = a * nkv // nh
        s = np.where(seen, q[:, a] @ k[g].T / np.sqrt(hd), -np.inf)
        e = np.exp(s - s.max(1, keepdims=True))
        want[a] = e / e.sum(1, keepdims=True) @ (v[g] if spoil is None else np.where(np.isfinite(v[g]), v[g], 0))
    return got, want


# a weight is off by 2^-11 of itself at most, and so is the result's norm under values that are independent of one another; what is left of twice that is for
# the correlation that chance gives a few hundred values
SHAPES = [(128, 4, 4, 0, 0, 17, 64), (128, 4, 4, 0, 0, 63, 64), (128, 4, 4, 0, 1, 64, 96), (128, 4, 2, 0, 63, 65, 160), (64, 8, 2, 2, 0, 127, 160), (64, 4, 4, 0, 64, 128, 192),
          (64, 8, 1, 2, 5, 129, 160), (128, 2, 2, 2, 1900, 90, 2400), (128, 2, 1, 0, 0, 700, 736), (64, 256, 8, 2, 30, 129, 160), (128, 256, 8, 0, 3, 190, 224)]


@pytest.mark.parametrize("hd,nh,nkv,mode,past,T,n_ctx", SHAPES + [(128, 4, 4, 0, 12500, 40, 14000)])
def test_matches_float64(hd, nh, nkv, mode, past, T, n_ctx):
    got, want = run(hd, nh, nkv, mode, past, T, n_ctx)
    for a, w in want.items():
        assert np.linalg.norm(got[:, a] - w) < 2.0 ** -10 * np.linalg.norm(w), a


@pytest.mark.parametrize("hd,T,past,grow", [(64, 130, 300, 40.0), (128, 200, 0, 12.0), (128, 40, 700, -40.0)])
def test_scores_that_keep_growing_or_falling(hd, T, past, grow):
    """Scores up to several hundred: a row's base is raised in most tiles (growing), or never after the first (falling: the first cell has 0).  A score of
    300 is off by 300 * 2^-24 * 1.5 times a few sums, which is next to nothing beside 2^-11."""
    got, want = run(hd, 2, 2, 0, past, T, past + T + 8, grow=grow)
    for a, w in want.items():
        assert np.isfinite(got[:, a]).all() and np.linalg.norm(got[:, a] - w) < 2.0 ** -10 * np.linalg.norm(w), a


@pytest.mark.parametrize("hd,T,spoil", [(128, 70, 40), (64, 150, 149), (128, 40, 0)])
def test_a_value_that_is_no_number_reaches_the_tokens_that_see_it_only(hd, T, spoil):
    got, want = run(hd, 2, 2, 0, 10, T, 192, spoil=spoil)
    for a, w in want.items():
        assert np.isfinite(got[:spoil, a]).all() and not np.isfinite(got[spoil:, a]).any()
        if spoil:
            assert np.linalg.norm(got[:spoil, a] - w[:spoil]) < 2.0 ** -10 * np.linalg.norm(w[:spoil])


def test_what_it_does_not_cover_is_refused():
    from powerinfer_amd import lib as pl
    L, b = pl.init(), pl.DevBuf(1 << 16)
    call = lambda hd, T, stride, off=0: L.pi_k_attn_chunk_once(b.ptr + off, 3 * hd, T, 1, 1, hd, 0, 0.9, 1.0, b.ptr, 64, 32, b.ptr, b.ptr, b.ptr, b.ptr, stride, None, None)  # noqa: E731
    assert call(32, 17, 32) != 0 and call(64, 17, 66) != 0 and call(64, 16, 64) != 0 and call(64, 17, 64, 4) != 0
