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
    # the groups' sums of squares run in another order: n squares' sums differ by n * 2^-24 of themselves at most, their roots by half of that; behind them sums of taps + 1
    # products of such inputs, and one rounding of the result
    off = cols // groups * 2.0 ** -24
    assert (np.abs(s1 - s2) <= off * np.abs(s1)).all()
    top = np.abs(x1).max() * 40                                       # (of a normed input times a weight)
    assert np.abs(h1 - h2).max() <= off * top * (taps + 1) + (2.0 ** -8 if t == pl.BF16 else 2.0 ** -22) * np.abs(h1).max()


def test_sizes_that_are_not_supported():
    L = pl.init()
    assert not L.pi_k_sum_conv_supported(4096, 32, 4, 4096, 12288) and not L.pi_k_sum_conv_supported(8192, 1, 4, 8192, 24576) and not L.pi_k_sum_conv_supported(4096, 8, 6, 4096, 20480)
