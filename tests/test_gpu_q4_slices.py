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
