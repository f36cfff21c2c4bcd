"""The last layer of prompts: sparse models keep only its keys and values for the tokens of a chunk."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,layers,hot", [("llama-tiny", 1, 1.0), ("llama-tiny", 3, 1.0), ("falcon-tiny", 1, 1.0), ("falcon-tiny", 2, 1.0), ("llama-tiny", 2, 0.6)])
@pytest.mark.parametrize("n", [3, 17, 18, 34, 131, 530])
def test_a_step_behind_a_prompt(name, layers, hot, n):
    """Logits of the step behind a prompt, whose cells a chunk wrote, against those behind the same tokens one by one: both are sums of the same fp16
    products in fp32, 1e-2 as for the CPU path."""
    from powerinfer_amd.model import Model
    hp = synth.hparams(name, n_layer=layers, n_rank=256, n_ctx=600, seed=13, pred_margin=True, hot_frac=hot)
    model = synth.make_model(hp)
    toks = np.random.default_rng(n).integers(0, hp.n_vocab, n).astype(np.int32)
    a, b = Model(hp).load(model), Model(hp).load(model)
    a.decode(toks, 0)
    for k, t in enumerate(toks):
        b.decode([t], k, want_logits=False)
    got, want = a.decode([7], n)[1], b.decode([7], n)[1]
    a.close()
    b.close()
    assert np.abs(got - want).max() < 1e-2 * np.abs(want).max()
