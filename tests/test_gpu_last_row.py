"""The token that ends an F16 prompt goes along in its last chunk and only through the last layer by itself."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu
SHAPES = [("llama-tiny", 1, 256), ("llama-tiny", 3, 256), ("llama-tiny", 3, 128), ("falcon-tiny", 2, 256)]
CASES = [s + (n,) for s in SHAPES for n in (3, 16, 17, 18, 33, 129, 530)] + [("llama-tiny", 2, 256, n) for n in (2048, 2049, 2050)]


@pytest.mark.parametrize("name,layers,rank,n", CASES)
def test_logits_counts_and_state_behind_a_prompt(name, layers, rank, n):
    """Against the same tokens one by one: both are sums of the same fp16 products in fp32, 1e-2 as for the CPU path; as many neurons fire for the last token
    (every decision has a margin), and the tokens generated from there on are the same."""
    from powerinfer_amd.model import Model
    hp = synth.hparams(name, n_layer=layers, n_ff=8192, n_rank=rank, n_ctx=max(600, n + 16), seed=13, pred_margin=True, head_pair=2048)
    model = synth.make_model(hp)
    toks = np.random.default_rng(n).integers(0, hp.n_vocab, n).astype(np.int32)
    a, b = Model(hp).load(model), Model(hp).load(model)
    first, got = a.decode(toks, 0)
    for k, t in enumerate(toks):
        again, want = b.decode([t], k)
    assert np.abs(got - want).max() < 1e-2 * np.abs(want).max()
    assert first == again and np.array_equal(a.step_active(1), b.step_active(1))
    assert np.array_equal(a.generate(8)[0], b.generate(8)[0])
    a.close()
    b.close()
