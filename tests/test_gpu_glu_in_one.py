"""Dense feed-forwards of long passes, whose gate, up and GLU are one product from 1400 tokens on where their rows need no padding, against the same prompt in
shorter passes."""
import numpy as np
import pytest

import fikevik_models as fm
from lerasun_models import row_errors, tokens
from powerinfer_amd import fikevik

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1399, 1400, 1537])
@pytest.mark.parametrize("ff", [128, 192, 256, 320, 384])
def test_long_passes_match_short_ones(n, ff):
    """Every wanted logit (17: no row is left out of the last layer) of one pass and of passes of 700 tokens: the products are the same, their sums in
    another order, and the activations round to bf16 in both, 2^-8 of a value; four times that of a row, and twice over the two layers."""
    cfg = fm.config(256, 200, [fm.gla(2, 64, 64, mlp=fm.dense(ff)), fm.gla(4, 32, 64, mlp=fm.dense(ff))])
    w, toks, out = fm.weights(cfg, 5), tokens(cfg, n, 3), []
    want = list(range(n - 17 * 40, n, 40))
    for batch in (2048, 700):
        m = fikevik.build(cfg, w, n_ctx=2048, max_batch=batch)
        m.kv_cells_init(2048)
        out.append(m.kv_cells_step(toks, range(n), [1] * n, want)[1])
        m.close()
    assert out[0].shape == (17, 200) and row_errors(out[0], out[1]).max() < 2 ** -5
