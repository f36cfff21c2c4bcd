"""F16 prompts around the length from which chunks of smaller layers go through a list of the neurons that fire for one of their tokens."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["llama-tiny", "falcon-tiny"])
def test_against_single_tokens(name):
    """Both are sums of the same fp16 products in fp32, 1e-2 as for the CPU path; as many neurons fire for the last token (every decision has a margin)."""
    from powerinfer_amd.model import Model
    hp = synth.hparams(name, n_layer=3, n_ff=8192, n_rank=256, n_ctx=300, seed=13, pred_margin=True, head_pair=2048)
    weights = synth.make_model(hp)
    toks = np.random.default_rng(1).integers(0, hp.n_vocab, 259).astype(np.int32)
    a, b = Model(hp).load(weights), Model(hp).load(weights)
    for k, t in enumerate(toks):
        tok, want = b.decode([t], k)
        if k + 1 in (128, 129, 130, 256, 257, 258, 259):
            first, got = a.decode(toks[:k + 1], 0)
            assert np.abs(got - want).max() < 1e-2 * np.abs(want).max(), k + 1
            assert first == tok and np.array_equal(a.step_active(1), b.step_active(1))
    a.close()
    b.close()
