"""The longest F16 chunks of layers with more than 48 million weights a matrix: the down projection goes by a copy of its matrix with the neurons contiguous where all of them fire, which the
host hears of in the middle of the layer, and over the listed rows otherwise."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["llama-tiny", "falcon-tiny"])
def test_against_shorter_chunks(name):
    """A prompt of one long chunk and the same one in two calls, of which neither is that long: sums of the same fp16 products in fp32, 1e-2 as for the CPU path.  All neurons fire
    (the first call makes the copy, the next ones find it), or those of the predictor's choice, with a margin."""
    from powerinfer_amd.model import Model
    d, ff, n = 2048, 24832, 1800
    hp = synth.hparams(name, n_layer=2, n_embd=d, n_head=16, n_head_kv=16 if name == "llama-tiny" else 2, n_ff=ff, n_rank=256, n_vocab=512, n_ctx=1900, seed=3, pred_margin=True, head_pair=2048)
    weights = synth.make_model(hp)
    toks = np.random.default_rng(1).integers(0, hp.n_vocab, n + 60).astype(np.int32)
    for threshold in (-1e30, hp.sparse_threshold):
        m = Model(synth.HParams(hp, sparse_threshold=threshold)).load(weights)
        m.decode(toks[:1000], 0, want_logits=False)
        tok, want = m.decode(toks[1000:n], 1000)
        for again in range(3):
            print(name, threshold, again, flush=True)
            first, got = m.decode(toks[:n], 0)
            assert np.abs(got - want).max() < 1e-2 * np.abs(want).max()
            assert first == tok
        m.close()
