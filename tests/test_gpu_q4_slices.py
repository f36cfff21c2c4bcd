"""Rows of Q4_0 matrices through LDS (q4_slice_fetch): groups of 32 neurons with none, few and all of them active - more than the eight whose rows
travel together - against the CPU reference, and matrices that do not start on a multiple of 16 bytes, bit for bit."""
import numpy as np
import pytest

import oracle_lib as ol
from powerinfer_amd import lib as pl
from powerinfer_amd import synth
from test_gpu_ffn import FFN_REL_TOL, rel_err, under

pytestmark = pytest.mark.gpu


class Shifted:
    """The bytes of a buffer two bytes behind a multiple of 16."""

    def __init__(self, buf):
        host = buf.download(np.uint8)
        self.buf = pl.DevBuf(host=np.concatenate([np.zeros(2, np.uint8), host, np.zeros(14, np.uint8)]))
        self.ptr = self.buf.ptr + 2


@pytest.mark.parametrize("has_gate,r,threshold", [(True, 1024, 0.0), (True, 512, -3e38), (False, 512, 0.0), (False, 1024, 3e38)])
def test_busy_groups_and_odd_addresses(has_gate, r, threshold):
    from powerinfer_amd.ops import SparseFFN
    d, ff = 4096, 1024
    L = synth.make_ffn_layer(seed=r, d=d, ff=ff, r=r, wtype=ol.Q4_0, has_gate=has_gate, mean_rate=0.4, T=1)
    x = np.ascontiguousarray(L["x"][:1], np.float32)
    out = []
    for shift in (False, True):
        ffn = SparseFFN(d, ff, r, ol.Q4_0, L["up"], L["gate"], L["down_t"], L["fc1"], L["fc2"], threshold=threshold)
        if shift:
            for name in ("up", "gate", "down"):
                if getattr(ffn, name) is not None:
                    setattr(ffn, name, Shifted(getattr(ffn, name)))
        print(has_gate, r, threshold, shift, flush=True)
        one = ffn.forward_q4_one_launch(x[0], x[0])
        two = ffn.forward_q4_fused(x[0], x[0])
        assert np.array_equal(one["h"], two["h"]) and rel_err(one["out"], two["out"]) < 1e-5 or not one["h"].any()
        out.append((one["h"], one["out"], two["out"]))
        n = np.add.reduceat((~(one["logits"] < threshold)).astype(int), np.arange(0, ff, 32))
        assert n.max() == (0 if threshold > 1e38 else 32) or (n.max() > 8 and n.min() < 20)
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    if threshold == 0.0:
        ou = under(L, d, ff, ol.Q4_0, has_gate, x, one["logits"])
        assert rel_err(out[0][0], ou["h"]) < 1e-4 and rel_err(out[0][1], ou["out"]) < FFN_REL_TOL


@pytest.mark.parametrize("has_gate,r,threshold", [(True, 1024, 0.0), (False, 512, -3e38)])
def test_rows_at_any_address(has_gate, r, threshold):
    """Up, gate and down matrices that start 4, 8, 12, 14 bytes behind a multiple of 16, at odd addresses, and each at another: the bits of aligned ones."""
    from powerinfer_amd.ops import SparseFFN

    class At:
        def __init__(self, buf, by):
            self.buf = pl.DevBuf(host=np.concatenate([np.zeros(by, np.uint8), buf.download(np.uint8), np.zeros(31 - by, np.uint8)]))
            self.ptr = self.buf.ptr + by

    d, ff = 4096, 512
    L = synth.make_ffn_layer(seed=r, d=d, ff=ff, r=r, wtype=ol.Q4_0, has_gate=has_gate, mean_rate=0.4, T=1)
    x, want = np.ascontiguousarray(L["x"][:1], np.float32)[0], None
    for at in ((0, 0, 0), (4, 4, 4), (8, 12, 14), (2, 0, 12), (14, 14, 0), (1, 1, 1), (15, 2, 0), (0, 4, 7)):
        ffn = SparseFFN(d, ff, r, ol.Q4_0, L["up"], L["gate"], L["down_t"], L["fc1"], L["fc2"], threshold=threshold)
        for name, by in zip(("up", "gate", "down"), at):
            if getattr(ffn, name) is not None:
                setattr(ffn, name, At(getattr(ffn, name), by))
        print(has_gate, r, at, flush=True)
        got = ffn.forward_q4_one_launch(x, x)
        want = want or got
        assert np.array_equal(got["h"], want["h"]) and np.array_equal(got["out"], want["out"]) and want["out"].any(), at


@pytest.mark.parametrize("rows,cols", [(5, 4096), (12290, 4096), (6145, 8192)])
def test_mat_vec_of_a_matrix_on_4_bytes(rows, cols):
    """Every multiple of 4 behind a multiple of 16: the bits of the aligned matrix."""
    L, rng, want = pl.init(), np.random.default_rng(rows), None
    raw = synth.quantize_q4_0((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)).reshape(-1).view(np.uint8)
    dx, y = pl.DevBuf(host=rng.standard_normal(cols).astype(np.float32)), pl.DevBuf(4 * rows)
    for off in (0, 4, 8, 12):
        dw = pl.DevBuf(host=np.concatenate([np.zeros(off, np.uint8), raw, np.zeros(16, np.uint8)]))
        print(rows, cols, off, flush=True)
        pl.check(L.pi_k_gemv(pl.Q4_0, dw.ptr + off, rows, cols, dx.ptr, None, pl.EPI_NONE, None, None, y.ptr, None))
        pl.sync()
        got = y.download(np.float32)
        want = got if want is None else want
        assert np.array_equal(got, want) and got.any(), off


@pytest.mark.parametrize("rows,cols,hot_frac", [(32, 4096, 1.0), (200, 256, 1.0), (72, 512, 1.0), (96, 4096, 0.6), (64, 8192, 0.0), (32, 96, 1.0), (160, 768, 0.3)])
@pytest.mark.parametrize("shift", [0, 2])
def test_expanded_matrices(rows, cols, hot_frac, shift):
    """A Q4_0 matrix as fp16, rows or columns contiguous, by units of 128 blocks and without them: exactly (q - 8) * d rounded to fp16."""
    L, rng = pl.init(), np.random.default_rng(rows + cols)
    wq = synth.quantize_q4_0((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    want = np.zeros((rows, cols), np.float32)
    ol.oracle().pio_dequantize_row_q4_0(ol._ptr(wq), ol._ptr(want), rows * cols)
    gid = rng.random(rows) < hot_frac
    words, prefix = None, None
    if hot_frac < 1.0:
        bits = np.packbits(gid.reshape(-1, 32), axis=1, bitorder="little").view(np.uint32).ravel()
        words, prefix = pl.DevBuf(host=bits), pl.DevBuf(host=np.concatenate([[0], np.cumsum(gid.reshape(-1, 32).sum(1))[:-1]]).astype(np.int32))
    place = lambda a: Shifted(pl.DevBuf(host=np.concatenate([a.reshape(-1).view(np.uint8), np.zeros(16, np.uint8)]))) if shift else pl.DevBuf(host=np.concatenate([a.reshape(-1).view(np.uint8), np.zeros(16, np.uint8)]))  # noqa: E731
    hot, rest = place(wq[gid] if words else wq), place(wq[~gid]) if words else None
    p = lambda b: b.ptr if b is not None else None  # noqa: E731
    for name, t in (("pi_k_dequant_q4_f16", False), ("pi_k_dequant_q4_t_f16", True)):
        out = pl.DevBuf(2 * rows * cols + 64)
        pl.check(L.pi_memset(out.ptr, 0xAB, out.nbytes))
        print(name, rows, cols, hot_frac, shift, flush=True)
        rc = getattr(L, name)(hot.ptr, p(rest), p(words), p(prefix), rows, cols, out.ptr, None)
        if t and (shift or cols % 256):
            assert rc != 0
            continue
        pl.check(rc, name)
        pl.sync()
        got = out.download(np.float16)
        assert (got[rows * cols:].view(np.uint16) == 0xABAB).all()
        assert np.array_equal(got[:rows * cols].reshape((cols, rows) if t else (rows, cols)), (want.T if t else want).astype(np.float16))


@pytest.mark.parametrize("rows,cols,kind", [(1, 4096, 0), (5, 4096, 1), (2047, 4096, 2), (2049, 4096, 0), (10241, 4096, 1), (12290, 4096, 0), (3, 8192, 1), (4100, 8192, 0), (6145, 8192, 2)])
def test_mat_vec_steps(rows, cols, kind):
    """Row counts around whole steps of the copying wave, one and two groups of 4096 columns: within 1e-5 of float64 over the same quantised
    input (128 or 256 fp32 terms a row), and the same bits for a matrix that starts on a multiple of 4 bytes only."""
    import ctypes as C
    from test_gpu_ffn import q4_rows_np, q8_blocks_np
    L, rng = pl.init(), np.random.default_rng(rows)
    wq = synth.quantize_q4_0((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    x, add = rng.standard_normal(cols).astype(np.float32), rng.standard_normal(rows).astype(np.float32)
    w, b = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32), (0.1 * rng.standard_normal(cols)).astype(np.float32)
    xn = x.copy()
    O, P = ol.oracle(), ol._ptr
    if kind == 1:
        O.pio_rms_norm(P(x), cols, 1, 1e-5, P(xn)); xn = np.ascontiguousarray(xn * w, np.float32)
    elif kind == 2:
        O.pio_norm(P(x), cols, 1, 1e-5, P(xn)); xn = np.ascontiguousarray(xn * w + b, np.float32)
    q, d = q8_blocks_np(xn)
    got = []
    raw = wq.reshape(-1).view(np.uint8)
    for off in (0, 4):
        dw = pl.DevBuf(host=np.concatenate([np.zeros(off, np.uint8), raw, np.zeros(16, np.uint8)]))
        dx, dn, db, da, y = pl.DevBuf(host=x), pl.DevBuf(host=w), pl.DevBuf(host=b), pl.DevBuf(host=add), pl.DevBuf(4 * rows + 64)
        pl.check(L.pi_memset(y.ptr, 0xAB, y.nbytes))
        nrm = pl.Norm(kind=kind, eps=1e-5, w=dn.ptr, b=db.ptr if kind == 2 else None) if kind else None
        print(rows, cols, kind, off, flush=True)
        pl.check(L.pi_k_gemv(pl.Q4_0, dw.ptr + off, rows, cols, dx.ptr, C.byref(nrm) if nrm else None, pl.EPI_ADD, da.ptr, None, y.ptr, None))
        pl.sync()
        out = y.download(np.float32)
        assert (out[rows:].view(np.uint32) == 0xABABABAB).all()
        got.append(out[:rows])
    assert np.array_equal(*got)
    v, s = q4_rows_np(raw.reshape(rows, -1), np.arange(rows), cols)
    sums = (v.reshape(rows, -1, 32) * q.reshape(1, -1, 32)).sum(2)
    want = (sums * s.astype(np.float64) * d.reshape(-1, 32)[:, 0]).sum(1)
    assert np.abs(got[0] - add - want).max() <= 1e-5 * max(np.abs(want).max(), np.abs(add).max())
