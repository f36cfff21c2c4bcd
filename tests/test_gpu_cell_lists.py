"""Cells of a step on their way into the sequences' lists: few travel as arguments of a kernel, more through a copy."""
import numpy as np
import pytest

from lerasun_models import odd_config, tokens, weights
from powerinfer_amd import lerasun, lib as pl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 21, 31, 32, 33, 64, 65])
def test_shared_cells_are_those_of_one_sequence(n):
    """Two sequences that share n cells (2 n entries of their lists) against one that owns them (n entries): what follows has the same bits, step by step,
    also where steps follow one another without a pause."""
    cfg = odd_config()
    w, p, after = weights(cfg, 17), tokens(cfg, n, 1), tokens(cfg, 3, 2)
    out = []
    for mask in (1, 3):
        m = lerasun.build(cfg, w, compute=pl.F32, n_ctx=128)
        m.kv_cells_init(128)
        m.kv_cells_step(p, range(n), [mask] * n, [], want_logits=False)
        out.append([m.kv_cells_step([t], [n + k], [1], [0])[1] for k, t in enumerate(after)])
        if mask == 3:
            out.append([m.kv_cells_step([t], [n + k], [2], [0])[1] for k, t in enumerate(after)])
        m.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("n", [70, 150, 300])
def test_a_step_whose_positions_go_back(n):
    """One sequence's tokens in one call, the second part of them ahead of the first: the logits are those of the call that has them in order.  A token's sums are the
    same either way (its cells in the order of their positions), so all that may differ is how the tokens are grouped: fp32 rounding."""
    cfg = odd_config()
    w, p = weights(cfg, 17), tokens(cfg, n, 1)
    turned = list(range(n // 3, n)) + list(range(n // 3))
    out = []
    for order in (list(range(n)), turned):
        m = lerasun.build(cfg, w, compute=pl.F32, n_ctx=512)
        m.kv_cells_init(512)
        logits = m.kv_cells_step([p[k] for k in order], order, [1] * n, list(range(n)))[1]
        out.append(np.asarray(logits)[np.argsort(order)])
        out.append(np.asarray(m.kv_cells_step([9], [n], [1], [0])[1]))
        m.close()
    for a, b in ((out[0], out[2]), (out[1], out[3])):
        assert np.abs(a - b).max() <= 1e-5 * np.abs(a).max()
