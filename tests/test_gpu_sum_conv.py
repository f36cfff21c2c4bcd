"""A layer's last sum with the next layer's norm and convolution in one launch: the results of the two operators, for fresh and continued runs of one to three tokens, one to five taps, both
layouts, groups of one wave and of sixteen."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_gqa_ops import filled
from test_gpu_latent_ops import TYPES, dev, fetch, i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("cols,groups,taps,ol", [(4096, 8, 4, 1), (256, 1, 1, 0), (4096, 1, 5, 0), (1536, 2, 2, 1), (512, 2, 3, 0)])
def test_as_in_two_launches(t, cols, groups, taps, ol):
    if ol and t == pl.F32:
        return
    L, rng = pl.init(), np.random.default_rng(cols + taps)
    most = L.pi_k_conv_tokens(7, taps)
    runs = [(min(n, most), fresh) for n, fresh in ((1, 0), (3, 1), (1, 1), (2, 0))]      # tokens, fresh
    T, slot_ld, ld = sum(n for n, _ in runs), (taps - 1) * cols + 8, cols + 64
    items, at = [], 0
    for slot, (n, fresh) in enumerate(runs):
        items.append([at, n, 0, n, len(runs) - 1 - slot, fresh, 0, 0])
        at += n
    x, mix = (rng.standard_normal((T, cols)).astype(np.float32) for _ in range(2))
    w1, w2 = ((1 + 0.3 * rng.standard_normal(cols)).astype(np.float32) for _ in range(2))
    taps_w, state = (0.5 * rng.standard_normal((taps, cols))).astype(np.float32), rng.standard_normal((len(runs), slot_ld)).astype(np.float32)
    mb, ab, bb, tb, ib = dev(mix), dev(w1), dev(w2), dev(taps_w), i32(items)
    assert L.pi_k_sum_conv_supported(cols, groups, taps, ld, slot_ld)
    got = []
    for one in (False, True):
        xb, sb, keep, h = dev(x), dev(state), pl.DevBuf.zeros(4 * T * cols), pl.DevBuf.zeros(4 * 16 * ld)
        p = filled(pl.SumNorm, x=xb, mix=mb, w=ab, mult=0.7, T=T, cols=cols, groups=groups, eps=1e-5, keep=keep, ld=ld, ol=ol)
        c = filled(pl.ConvNorm, x=xb, w=bb, taps_w=tb, T=T, cols=cols, groups=groups, taps=taps, eps=1e-5, state=sb, slot_ld=slot_ld, items=ib, n_items=len(items), h=h, ld=ld, ol=ol)
        print(t, cols, groups, taps, ol, one, flush=True)
        if one:
            pl.check(L.pi_k_sum_conv(t, C.byref(p), C.byref(c), None))
        else:
            pl.check(L.pi_k_sum_norm(t, C.byref(p), None))
            pl.check(L.pi_k_conv_norm(t, C.byref(c), None))
        pl.sync()
        got.append([xb.download(np.float32), keep.download(np.float32), sb.download(np.float32), fetch(h, t, (ld // 8, 16, 8)) if ol else fetch(h, t, (T, ld))[:, :cols]])
    (x1, k1, s1, h1), (x2, k2, s2, h2) = got
    assert np.array_equal(x1, x2) and np.array_equal(k1, k2)
    # The groups' sums of squares run in another order: a chain of at most size / 64 additions of a lane (four squares of every 256 columns), 6 of a wave and 16 of the waves, so that two of
    # them are within that many 2^-24 of the squares' sum on either side, and their roots within half of both together.  Two roundings behind it for an input; an output is
    # taps + 1 products of inputs (the last one's tap and itself), a rounding each, and one of the result in bf16 that may fall the other way.
    size = cols // groups
    off = (size / 64 + 22 + 4) * 2.0 ** -24
    assert (np.abs(s1 - s2) <= off * np.abs(s1)).all()
    rows = lambda h: h.transpose(1, 0, 2).reshape(16, ld)[:T, :cols] if ol else h      # noqa: E731
    u = x1.reshape(T, groups, size).astype(np.float64)
    u = (u / np.sqrt((u ** 2).mean(-1, keepdims=True) + 1e-5)).reshape(T, cols) * w2
    for (first, n, _, _, slot, fresh, _, _) in items:
        past = np.zeros((taps - 1, cols)) if fresh else state[slot, :(taps - 1) * cols].reshape(taps - 1, cols)
        run = np.abs(np.concatenate([past, u[first:first + n]]))
        for k in range(n):
            terms = run[taps - 1 + k] + (np.abs(taps_w) * run[k:k + taps]).sum(0)
            a, b = rows(h1)[first + k], rows(h2)[first + k]
            assert (np.abs(a - b) <= (off + (taps + 1) * 2.0 ** -24) * terms + (2.0 ** -7 * np.abs(a) if t == pl.BF16 else 0)).all()
            want = u[first + k] + (taps_w * np.concatenate([past, u[first:first + n]])[k:k + taps]).sum(0)
            assert (np.abs(b - want) <= (off + (taps + 1) * 2.0 ** -24) * terms + (2.0 ** -8 * np.abs(want) if t == pl.BF16 else 0)).all()


def test_sizes_that_are_not_supported():
    L = pl.init()
    assert not L.pi_k_sum_conv_supported(4096, 32, 4, 4096, 12288) and not L.pi_k_sum_conv_supported(8192, 1, 4, 8192, 24576) and not L.pi_k_sum_conv_supported(4096, 8, 6, 4096, 20480)
