"""A token's embedding row formed by the mat-vec that reads it: the row, the products and the loop's state bit for bit those of the two launches, at the widths of every kernel that
takes it, rows that do not fill a workgroup, matrices on 16 and on 4 bytes, tokens named by the host and by the device; refused at the widths around them."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [1, 2])
@pytest.mark.parametrize("wtype,rows,cols,off", [(pl.F16, 1536, 512, 0), (pl.F16, 7, 8, 0), (pl.F16, 301, 1016, 0), (pl.F16, 3072, 1024, 0), (pl.F16, 5000, 4096, 0), (pl.F16, 4097, 5120, 0),
                                                 (pl.F16, 2050, 8192, 0), (pl.Q4_0, 4099, 4096, 0), (pl.Q4_0, 2050, 8192, 4), (pl.Q4_0, 3, 4096, 8)])
def test_first_gemv(wtype, rows, cols, off, kind):
    L, rng, vocab = pl.init(), np.random.default_rng(rows + cols), 37
    make = (lambda n: (rng.standard_normal((n, cols)) * 0.3).astype(np.float16)) if wtype == pl.F16 else (lambda n: synth.quantize_q4_0((rng.standard_normal((n, cols)) * 0.3).astype(np.float32)))
    table, W = pl.DevBuf(host=make(vocab)), make(rows)
    dw = pl.DevBuf(host=np.concatenate([np.zeros(off, np.uint8), np.ascontiguousarray(W).view(np.uint8).ravel()]))
    w, b = (pl.DevBuf(host=rng.standard_normal(cols).astype(np.float32)) for _ in range(2))
    n = pl.Norm(kind, 1e-5, w.ptr, b.ptr if kind == 2 else None)
    xs, ys = [[pl.DevBuf(host=np.full(k, 7, np.float32)) for _ in range(2)] for k in (cols, rows)]
    state = pl.DevBuf(host=np.array([5, 6, 7], np.int32))
    assert L.pi_k_first_gemv_supported(wtype, table.ptr, dw.ptr + off, rows, cols, C.byref(n), xs[0].ptr) == 1
    for token in (0, vocab - 1, 11):
        print(wtype, rows, cols, off, kind, token, flush=True)
        named = pl.DevBuf(host=np.array([token], np.int32))
        pl.check(L.pi_k_embed(wtype, table.ptr, cols, named.ptr, xs[0].ptr, None))
        pl.check(L.pi_k_gemv(wtype, dw.ptr + off, rows, cols, xs[0].ptr, C.byref(n), 0, None, None, ys[0].ptr, None))
        want = xs[0].download(np.float32), ys[0].download(np.float32)
        for by_host in (False, True):
            before = state.download(np.int32).tolist()
            at = [state.ptr + 4 * k if by_host else None for k in range(3)]
            pl.check(L.pi_k_first_gemv(wtype, table.ptr, None if by_host else named.ptr, token, 100 + token, *at, dw.ptr + off, rows, cols, C.byref(n), xs[1].ptr, ys[1].ptr, None))
            np.testing.assert_array_equal(xs[1].download(np.float32), want[0])
            np.testing.assert_array_equal(ys[1].download(np.float32), want[1])
            assert state.download(np.int32).tolist() == ([token, 100 + token, 0] if by_host else before)


def test_refusals():
    L, at = pl.init(), 4096                            # (addresses that nothing reads)
    n = pl.Norm(1, 1e-5, at, None)
    ok = lambda t, cols, n=n, table=at, W=at, x=at: L.pi_k_first_gemv_supported(t, table, W, 64, cols, C.byref(n), x)
    assert ok(pl.F16, 1024) and ok(pl.Q4_0, 4096)
    assert not any([ok(pl.F16, 1032), ok(pl.F16, 1020), ok(pl.F16, 2048), ok(pl.Q4_0, 512), ok(pl.Q4_0, 5120), ok(pl.F32, 512), ok(pl.F16, 512, table=at + 2), ok(pl.F16, 512, x=at + 4),
                    ok(pl.Q4_0, 4096, W=at + 2), ok(pl.F16, 512, pl.Norm(0, 0.0, None, None)), ok(pl.F16, 512, pl.Norm(1, 1e-5, at, at)), ok(pl.F16, 512, pl.Norm(2, 1e-5, at, None))])
