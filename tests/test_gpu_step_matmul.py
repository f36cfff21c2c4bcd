"""Mat-muls of steps of up to 16 tokens where the rows of a workgroup and the columns it starts with change (pi_k_gemm_f16_ol)."""
import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(5120, 256), (5120, 1024), (5121, 2048), (8193, 2048), (8224, 4096), (12256, 4096), (12288, 4096), (6144, 4096), (40, 8192), (5136, 8192), (5120, 5120),
                                       (8200, 512), (1024, 16384), (5130, 12288), (5120, 1280)])
@pytest.mark.parametrize("T", [1, 3, 16])
def test_against_sums_in_64_bits(rows, cols, T):
    """Around one workgroup of 32 rows for every compute unit and one and a half, short and long rows, rows whose starts are and are not 256 KB apart, fewer
    and more super-steps than waves.  A sum of n products in fp32 is off by at most n 2^-24 of the sum of their magnitudes."""
    rng = np.random.default_rng(rows + cols + T)
    w, x = rng.standard_normal((rows, cols)).astype(np.float16), rng.standard_normal((T, cols)).astype(np.float16)
    xo = np.zeros((cols // 8, 16, 8), np.float16)
    xo[:, :T] = x.reshape(T, cols // 8, 8).transpose(1, 0, 2)
    L = pl.init()
    dw, dx, dy = pl.DevBuf(host=w), pl.DevBuf(host=xo), pl.DevBuf(host=np.full((T, rows), np.nan, np.float32))
    pl.check(L.pi_k_gemm_f16_ol(dw.ptr, rows, cols, dx.ptr, T, pl.EPI_NONE, None, None, dy.ptr, None, None), "gemm")
    pl.sync()
    got = dy.download(np.float32).reshape(T, rows)
    W, X = w.astype(np.float64), x.astype(np.float64)
    assert (np.abs(got - X @ W.T) <= cols * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T)).all()
