"""One token's attention with a head's cells split over workgroups (attn_part_kernel, attn_merge_kernel) against float64 with the kernel's rounding points: s - m
of a part's maximum m and its exponential to fp16.  Numbers of cells around a part's batches (4 cells of each of 4096 / hd groups, two of them in
flight), parts without cells, every way a head's lanes may lie."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def attend(hd, nh, nkv, parts, n_kv, n_ctx, cached, spread=1.0):
    from powerinfer_amd import lib as pl
    L = pl.init()
    rng = np.random.default_rng(hd + parts + n_kv)
    d, gqa, n_seq = nh * hd, nkv * hd, 2
    qkv = (rng.standard_normal((n_seq, d + 2 * gqa)) * spread).astype(np.float32)
    kc, vc = rng.standard_normal((n_seq, nkv, n_ctx, hd)).astype(np.float16), rng.standard_normal((n_seq, nkv, n_ctx, hd)).astype(np.float16)
    kc[:, :, n_kv:], vc[:, :, n_kv:] = np.nan, np.nan
    if not cached:
        kc[:, :, n_kv - 1], vc[:, :, n_kv - 1] = np.nan, np.nan            # the new cell, not there yet
    table = np.zeros((n_ctx, hd // 2, 2), np.float32)
    table[..., 0] = 1                                                       # nothing is turned
    dq, dk, dv, tab, pos = (pl.DevBuf(host=a) for a in (np.ascontiguousarray(qkv[:, :d]) if cached else qkv, kc, vc, table, np.full(n_seq, n_kv - 1, np.int32)))
    out, scr = pl.DevBuf(n_seq * d * 4), pl.DevBuf(4 * L.pi_k_attn_split_scratch_floats(n_seq, nh, hd, parts))
    print("split", hd, nh, nkv, parts, n_kv, cached, flush=True)
    got, want, q = [], [], qkv[:, :d].astype(np.float16).astype(np.float64).reshape(n_seq, nh, hd)
    if cached:                                                              # both tokens on the first cache
        pl.check(L.pi_k_attn_split_cached(dq.ptr, dk.ptr, dv.ptr, n_seq, nh, nkv, hd, n_ctx, parts, pos.ptr, scr.ptr, out.ptr, None), "cached")
        k, v = kc[[0, 0], :, :n_kv].astype(np.float64), vc[[0, 0], :, :n_kv].astype(np.float64)
    else:
        pl.check(L.pi_k_attn_split(dq.ptr, d + 2 * gqa, tab.ptr, dk.ptr, dv.ptr, nkv * n_ctx * hd, n_seq, nh, nkv, hd, 0, n_ctx, parts, pos.ptr, scr.ptr, out.ptr, d, None, None), "split")
        pl.sync()
        for buf, cache, at in ((dk, kc, d), (dv, vc, d + gqa)):
            cache[:, :, n_kv - 1] = qkv[:, at:at + gqa].reshape(n_seq, nkv, hd).astype(np.float16)
            assert np.array_equal(buf.download(np.float16).reshape(cache.shape), cache, equal_nan=True)
        k, v = kc[:, :, :n_kv].astype(np.float64), vc[:, :, :n_kv].astype(np.float64)
    pl.sync()
    got = out.download(np.float32).reshape(n_seq, nh, hd)
    want = np.empty((n_seq, nh, hd))
    for b in range(n_seq):
        for h in range(nh):
            s = (k[b, h * nkv // nh] @ q[b, h] / np.sqrt(hd)).astype(np.float32)
            e, at = np.empty(n_kv), [n_kv * p // parts for p in range(parts + 1)]
            for lo, hi in zip(at, at[1:]):
                if hi > lo:
                    x = (s[lo:hi] - s[lo:hi].max()).astype(np.float16).astype(np.float64)
                    e[lo:hi] = np.exp(x).astype(np.float16).astype(np.float64) * np.exp(float(s[lo:hi].max()) - float(s.max()))
            want[b, h] = e @ v[b, h * nkv // nh] / e.sum()
    return got, want


@pytest.mark.parametrize("cached", [False, True])
@pytest.mark.parametrize("hd,nh,nkv,parts,n_kv", [(128, 4, 2, 1, n) for n in (1, 2, 127, 128, 129, 130, 255, 256, 257, 384, 385, 700)] + [
    (64, 4, 1, 3, n) for n in (1, 2, 3, 4, 767, 770, 1539, 2400)] + [(32, 4, 4, 5, 3000), (256, 2, 1, 16, 1000), (16, 2, 2, 2, 2055), (8, 4, 2, 1, 4097), (128, 2, 2, 64, 900)])
def test_matches_float64(hd, nh, nkv, parts, n_kv, cached):
    """A score of a few units is off by 2^-24 of itself a few times and so falls to the other side of an fp16 rounding in one cell of a few hundred, which moves
    that weight by 2^-10 of itself at most (s - m below 4 or its exponential): 2^-10 / sqrt(200) of the output; where the output is one cell's, of all of it."""
    got, want = attend(hd, nh, nkv, parts, n_kv, 4200, cached)
    assert np.linalg.norm(got - want) < (1e-4 if n_kv > 100 else 2.0 ** -10) * np.linalg.norm(want)


def test_scores_far_apart():
    """Scores in the hundreds: weights of one and of nothing; s - m of up to 16, which count, to fp16 units of 2^-7."""
    got, want = attend(128, 4, 4, 4, 900, 1000, False, spread=60.0)
    assert np.linalg.norm(got - want) < 2.0 ** -7 * np.linalg.norm(want)
