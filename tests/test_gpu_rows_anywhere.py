"""The sparse FFN of 8192 columns whose workgroups take several groups of neurons: a predictor matrix off a multiple of 16 bytes gives the bits of one on it, with the workspace's room and with the
8 MB of the call that allocates nothing."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [512, 1024])
@pytest.mark.parametrize("gate", [False, True])
def test_predictor_rows_anywhere(r, gate):
    L, rng = pl.init(), np.random.default_rng(r)
    ff, cols = 32768, 8192
    few = (rng.standard_normal((64, cols)) * 0.05).astype(np.float16)
    rows = [pl.DevBuf(host=np.tile(few, (ff // 64, 1)))]
    rows += [rows[0], rows[0]]
    fc2 = (rng.standard_normal((ff, r)) * r ** -0.5).astype(np.float16)
    fc2[:, 0] -= np.float16(1.5)                                  # (hidden unit 0 is positive: about a tenth fire)
    hidden = np.abs(rng.standard_normal(r)).astype(np.float32)
    x, w, b = (rng.standard_normal(cols).astype(np.float32) for _ in range(3))
    dh, dx, dw, db = (pl.DevBuf(host=v) for v in (hidden, x, w, b))
    nrm = pl.Norm(2, 1e-5, dw.ptr, db.ptr)
    ws = L.pi_workspace_create(ff, cols)
    got = []
    for off in (0, 4, 8):
        buf = pl.DevBuf(ff * r * 2 + 16)
        buf.upload(fc2, off)
        args = (buf.ptr + off, ff, r, dh.ptr, 0.0, rows[0].ptr, rows[1].ptr if gate else None, rows[2].ptr, cols, dx.ptr, C.byref(nrm), 0, None, None)
        for noalloc in (False, True):
            out, n = pl.DevBuf.zeros(cols * 4), pl.DevBuf.zeros(4)
            print(r, gate, off, noalloc, flush=True)
            if noalloc:
                pl.check(L.pi_k_sparse_ffn_noalloc(*args, out.ptr, None, None, n.ptr, None), "noalloc")
            else:
                pl.check(L.pi_k_sparse_ffn(*args, out.ptr, None, None, n.ptr, ws, None), "ffn")
            pl.sync()
            got.append((out.download(np.float32), int(n.download(np.int32)[0])))
    L.pi_workspace_destroy(ws)
    assert 0 < got[0][1] < ff and np.isfinite(got[0][0]).all() and np.abs(got[0][0]).max() > 0
    assert all(k == got[0][1] and np.array_equal(o, got[0][0]) for o, k in got)
