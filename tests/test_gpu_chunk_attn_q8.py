"""Attention of Q4_0 prompt chunks that leaves its output in blocks of eight bits: the bits of the two launches it replaces, by rows and in the operand layout, at edges of
the tiles of 16 tokens, both head sizes, grouped heads; refused where tokens are taken one by one."""
import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv,mode,past,T,n_ctx", [(128, 4, 4, 0, 0, 2, 64), (128, 8, 2, 2, 3, 16, 96), (64, 8, 8, 0, 40, 17, 128), (128, 32, 32, 0, 0, 130, 256), (64, 16, 1, 2, 600, 47, 700)])
def test_same_bits_as_in_two_launches(hd, nh, nkv, mode, past, T, n_ctx):
    L, rng = pl.init(), np.random.default_rng(hd + T)
    d, gqa, theta = nh * hd, nkv * hd, float(np.float32(10000.0) ** np.float32(-2.0 / hd))
    kc, vc = (rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16) for _ in range(2))
    qkv, pos = rng.standard_normal((T, d + 2 * gqa)).astype(np.float32), np.arange(past, past + T, dtype=np.int32)
    dq, dpos, rot, out = pl.DevBuf(host=qkv), pl.DevBuf(host=pos), pl.DevBuf(T * d * 4), pl.DevBuf(T * d * 4)
    slots = (T + 15) // 16 * 16
    for ol in (0, 1):
        got = []
        for one in (0, 1):
            dk, dv, h = pl.DevBuf(host=kc), pl.DevBuf(host=vc), pl.DevBuf(host=np.full(slots * d, np.nan, np.float16))
            print(hd, nh, nkv, past, T, ol, one, flush=True)
            if one:
                pl.check(L.pi_k_attn_chunk_q8(dq.ptr, d + 2 * gqa, T, nh, nkv, hd, mode, theta, 1.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, d, h.ptr, ol, None))
            else:
                pl.check(L.pi_k_attn_chunk(dq.ptr, d + 2 * gqa, T, nh, nkv, hd, mode, theta, 1.0, dpos.ptr, n_ctx, past + T, rot.ptr, dk.ptr, dv.ptr, out.ptr, d, None, None))
                f = L.pi_k_norm_q8_round_f16_ol if ol else L.pi_k_norm_q8_round_f16
                pl.check(f(out.ptr, T, d, None, h.ptr, None, None))
            pl.sync()
            got.append(h.download(np.float16))
        assert np.array_equal(got[0], got[1], equal_nan=True) and np.isfinite(got[1]).sum() == T * d


def test_refused_one_by_one():
    L = pl.init()
    b = pl.DevBuf.zeros(1 << 20)
    call = lambda T, hd: L.pi_k_attn_chunk_q8(b.ptr, 3 * hd, T, 1, 1, hd, 0, 0.9, 1.0, b.ptr, 64, 64, b.ptr, b.ptr, b.ptr, hd, b.ptr, 0, None)  # noqa: E731
    assert call(1, 128) != 0 and call(4, 96) != 0 and call(4, 32) != 0
