"""Kernels that read rows 16 bytes at a time against the ones for rows that do not start on a multiple of 16: RoPE and store of a prompt chunk, bit for
bit; the norm in front of the mat-muls, both against float64."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


def shifted(host, by):
    """A device copy that starts `by` bytes behind a multiple of 16."""
    raw = np.zeros(host.nbytes + 16, np.uint8)
    raw[by:by + host.nbytes] = host.view(np.uint8).ravel()
    buf = pl.DevBuf(host=raw)
    return buf, buf.ptr + by


@pytest.mark.parametrize("hd,nh,nkv,mode,T", [(8, 3, 1, 2, 17), (8, 2, 2, 0, 17), (64, 5, 5, 2, 130), (128, 4, 2, 0, 130), (32, 7, 7, 0, 63), (128, 48, 12, 0, 512), (64, 100, 4, 2, 512), (128, 32, 32, 2, 20)])
def test_rope_of_a_chunk(hd, nh, nkv, mode, T):
    L, rng = pl.init(), np.random.default_rng(hd + nh + T)
    width, n_ctx, past = (nh + 2 * nkv) * hd, T + 9, 5
    qkv = rng.standard_normal((T, width)).astype(np.float32)
    pos = pl.DevBuf(host=np.arange(past, past + T, dtype=np.int32))
    cells = rng.standard_normal((nkv, n_ctx, hd)).astype(np.float16)
    got = []
    for by in (0, 4):
        keep, ptr = shifted(qkv, by)
        k, v, rot, out = pl.DevBuf(host=cells), pl.DevBuf(host=cells), pl.DevBuf.zeros(T * nh * hd * 4), pl.DevBuf.zeros(T * nh * hd * 4)
        print(hd, nh, nkv, mode, T, by, flush=True)
        pl.check(L.pi_k_attn_chunk(ptr, width, T, nh, nkv, hd, mode, float(10000.0 ** (-2.0 / hd)), 1.0, pos.ptr, n_ctx, past + T, rot.ptr, k.ptr, v.ptr, out.ptr, nh * hd, None, None), "attn_chunk")
        got.append([b.download(np.uint8) for b in (rot, k, v, out)])
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    k16 = got[0][1].view(np.float16).reshape(nkv, n_ctx, hd)
    assert np.array_equal(k16[:, :past], cells[:, :past]) and np.array_equal(k16[:, past + T:], cells[:, past + T:])          # the chunk's cells only


@pytest.mark.parametrize("T,cols", [(1, 4), (3, 8), (2, 1020), (2, 1024), (2, 1028), (5, 4096), (2, 8188), (2, 8192), (1, 8196), (2, 6)])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("by", [0, 4])
def test_norm_of_rows(T, cols, kind, by):
    L, rng = pl.init(), np.random.default_rng(T + cols + kind)
    x = (rng.standard_normal((T, cols)) + 0.5).astype(np.float32)
    w, b = rng.standard_normal((2, cols)).astype(np.float32)
    (kx, px), dw, db = shifted(x, by), pl.DevBuf(host=w), pl.DevBuf(host=b)
    nrm = pl.Norm(kind, 1e-5, dw.ptr, db.ptr if kind == 2 else None)
    y = x.astype(np.float64)
    if kind == 2:
        y = y - y.mean(1, keepdims=True)
    if kind:
        y = y / np.sqrt((y * y).mean(1, keepdims=True) + 1e-5) * w + (b if kind == 2 else 0)
    # half a unit of fp16, and of the fp32 steps before it four of 2^-24 of the largest term (subnormal fp16: 2^-25)
    bound = np.abs(y) * 2.0 ** -11 + (np.abs(x).max() + 2) * (np.abs(w) + 1) * 2.0 ** -21 + 2.0 ** -25
    for ol in ([False, True] if cols % 8 == 0 else [False]):
        out, plain = pl.DevBuf.zeros(max(T, 16) * cols * 2), pl.DevBuf.zeros(max(T, 16) * cols * 2)
        print(T, cols, kind, by, ol, flush=True)
        pl.check((L.pi_k_norm_round_f16_ol if ol else L.pi_k_norm_round_f16)(px, T, cols, C.byref(nrm) if kind else None, out.ptr, plain.ptr, None), "norm")
        o, p = (a.download(np.float16) for a in (out, plain))
        o, p = (a.reshape(cols // 8, 16, 8).transpose(1, 0, 2).reshape(16, cols)[:T] if ol else a[:T * cols].reshape(T, cols) for a in (o, p))
        assert np.array_equal(p, x.astype(np.float16)) and (np.abs(o - y) <= bound).all()
