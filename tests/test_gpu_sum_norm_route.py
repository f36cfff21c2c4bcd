"""The norms between two sublayers with the expert choice behind them in one launch, against the three operators they are otherwise: up to 16 tokens, few and
many experts, one expert, all of them chosen, with a copy kept and without; the counters are back at zero and a second call finds them so."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl
from test_gpu_gqa_ops import filled
from test_gpu_latent_ops import dev, fetch, store

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups,size", [(8, 512), (1, 512), (3, 1024), (32, 512), (2, 1024)])
@pytest.mark.parametrize("E,top", [(64, 6), (1, 1), (7, 7), (63, 4), (128, 8)])
@pytest.mark.parametrize("T", [1, 5, 16])
def test_norms_and_choice(T, groups, size, E, top):
    if E * size > 65536:
        assert not pl.init().pi_k_sum_norm_route_supported(T, groups * size, groups, E)
        return
    L, rng = pl.init(), np.random.default_rng(T + groups + E)
    cols, ld = groups * size, groups * size + 128
    x, mix = (rng.standard_normal((T, cols)).astype(np.float32) for _ in range(2))
    w, w2 = ((1 + 0.3 * rng.standard_normal(cols)).astype(np.float32) for _ in range(2))
    router = np.zeros((E, ld), np.float32)
    router[:, :cols] = rng.standard_normal((E, cols))
    rb, mb, wb, w2b, sums, arrived = store(router, pl.BF16), dev(mix), dev(w), dev(w2), dev(np.zeros(T * groups * E)), pl.DevBuf.zeros(64)
    for _ in range(2):
        got = []
        for fused in (False, True):
            xb, keep, h = dev(x), pl.DevBuf.zeros(4 * T * cols), pl.DevBuf.zeros(2 * 16 * ld)
            z, ids, wts = pl.DevBuf.zeros(4 * T * E), pl.DevBuf.zeros(4 * T * top), pl.DevBuf.zeros(4 * T * top)
            p = filled(pl.SumNorm, x=xb, mix=mb, w=wb, mult=0.7, w_next=w2b, T=T, cols=cols, groups=groups, eps=1e-5, keep=keep, h=h, ld=ld, ol=1)
            print(T, groups, size, E, top, fused, flush=True)
            if fused:
                pl.check(L.pi_k_sum_norm_route(C.byref(p), rb.ptr, ld, E, top, ids.ptr, wts.ptr, sums.ptr, arrived.ptr, None))
            else:
                pl.check(L.pi_k_sum_norm(pl.BF16, C.byref(p), None))
                pl.check(L.pi_k_gemm_bf16_ol(rb.ptr, E, ld, h.ptr, T, pl.EPI_NONE, None, None, z.ptr, None, None))
                pl.check(L.pi_k_route_scores(z.ptr, T, E, top, ids.ptr, wts.ptr, None))
            pl.sync()
            got.append([xb.download(np.float32), keep.download(np.float32), fetch(h, pl.BF16, (ld // 8, 16, 8))[:, :T], ids.download(np.int32).reshape(T, top), wts.download(np.float32).reshape(T, top),
                        z.download(np.float32).reshape(T, E)])
        (x1, k1, h1, i1, w1, z1), (x2, k2, h2, i2, w2_, _) = got
        assert np.array_equal(x1, x2) and np.array_equal(k1, k2) and np.array_equal(x2, k2) and np.array_equal(h1, h2)
        # the scores differ by two orders of a sum of `cols` products of |h| |r|: no more than cols * 2^-24 of their magnitudes each; choices only among such
        hh = h2.transpose(1, 0, 2).reshape(T, ld)[:, :cols].astype(np.float64)
        off = 2 * cols * 2.0 ** -24 * (np.abs(hh) @ np.abs(fetch(rb, pl.BF16, (E, ld))[:, :cols].astype(np.float64)).T)
        for t in range(T):
            assert len(set(i2[t])) == top
            near = np.abs(z1[t][i2[t]] - z1[t][i1[t]]) <= off[t][i1[t]] + off[t][i2[t]]
            assert near.all() and (np.abs(w2_[t] - 1.0 / (1.0 + np.exp(-z1[t][i2[t]].astype(np.float64)))) <= off[t][i2[t]] + 1e-6).all()
        assert (arrived.download(np.int32) == 0).all()
