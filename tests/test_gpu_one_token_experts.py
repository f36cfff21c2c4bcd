"""One token's experts by streams of rows: first matrices of 2048, 4096 and 8192 columns, with fewer rows than workgroups, experts that end within a
workgroup's rows, sizes of 2048 columns that go in tiles, and beside the launch's other parts - the operators' own comparisons at these sizes."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_gqa_ops
import test_gpu_latent_ops
import test_gpu_layer_out
import test_gpu_pufivik_ops
from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,top,ff,cols,what", [(3, 2, 5, 2048, "gate"), (9, 6, 333, 4096, "both"), (2, 1, 514, 8192, "none"), (8, 8, 1027, 2048, "merge"), (8, 8, 1501, 2048, "merge"), (1, 1, 1, 4096, "none")])
def test_beside_merges_and_gates(E, top, ff, cols, what):
    test_gpu_gqa_ops.test_step_launch_beside_the_experts(1, E, top, ff, cols, what)


@pytest.mark.parametrize("E,top,ff,cols", [(7, 6, 171, 4096), (4, 3, 700, 2048), (4, 3, 1361, 2048), (3, 2, 65, 8192)])
def test_weighted_at_their_input(E, top, ff, cols):
    test_gpu_pufivik_ops.test_experts_of_a_step(1, E, top, ff, cols)


@pytest.mark.parametrize("E,top,ff,D", [(5, 3, 403, 2048), (5, 3, 2403, 2048), (4, 4, 129, 4096)])
def test_squared_beside_values(E, top, ff, D):
    test_gpu_latent_ops.test_step_kernels(1, 4, 16, 8, 24, 40, E, top, ff, D, 4)


@pytest.mark.parametrize("rows,ld_att,E,top,ld_act", [(4096, 0, 8, 6, 1408), (2048, 4864, 7, 6, 1408), (5120, 4096, 3, 2, 32), (1, 4096, 0, 0, 0), (257, 4128, 0, 0, 0), (4099, 8192, 9, 8, 2048), (100, 0, 1, 1, 32),
                                                        (16000, 512, 2, 2, 96), (17000, 512, 2, 2, 96), (300, 20480, 0, 0, 0), (300, 20512, 2, 2, 4096), (1, 4160, 0, 0, 0), (16000, 4064, 2, 2, 32),
                                                        (2049, 2048, 3, 2, 1024)])
def test_closing_a_layer(rows, ld_att, E, top, ld_act):
    """One to six pieces a thread and more than that, up to as many rows as a workgroup takes and more, parts of a last piece."""
    test_gpu_layer_out.test_closing_a_layer(rows, ld_att, E, top, ld_act, 1)


@pytest.mark.parametrize("ld_att", [4128, 8192, 12320])
def test_infinite_weights_close_a_layer(ld_att):
    """Threads without a last piece of their own hold it again: an infinite weight there is one term of its row's sum and no zero times infinity."""
    L, rng, rows = pl.init(), np.random.default_rng(ld_att), 4100
    wo, att = test_gpu_layer_out.bf16(rng.standard_normal((rows, ld_att))), test_gpu_layer_out.bf16(0.5 + rng.random((1, ld_att)))
    wo[7, ld_att - 1], wo[rows - 1, ld_att - 8] = test_gpu_layer_out.bf16([np.inf, -np.inf])
    w, a, out, s = pl.DevBuf(host=wo), pl.DevBuf(host=att), pl.DevBuf.zeros(4 * rows), pl.LayerOut()
    s.wo, s.att, s.ld_att, s.rows, s.T, s.out = w.ptr, a.ptr, ld_att, rows, 1, out.ptr
    pl.check(L.pi_k_layer_out_step(C.byref(s), None))
    got = out.download(np.float32)
    assert got[7] == np.inf and got[-1] == -np.inf and np.isfinite(np.delete(got, [7, rows - 1])).all()
