"""A small model's attention and output projection in one launch, the heads' shares added in front of the FFN: against the launches one by one that a capturing model takes."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,heads,kv_heads,rank,ff", [(512, 8, 8, 128, 4096), (512, 4, 2, 64, 96), (512, 8, 1, 256, 1024), (1024, 16, 4, 128, 4128), (1024, 8, 8, 64, 32)])
def test_decode_of_small_layers(d, heads, kv_heads, rank, ff):
    """Heads of 64 and 128, as many shares as a wave requests together and more, few cells and the last of the context.  Both sides round att, the probabilities and h to fp16 at the same
    places and sum in fp32 in another order, so that a value may round to the neighbouring fp16 number: 2^-11 of it, over three layers 2e-3 of the largest of 2048 logits.  Every decision
    of the predictor has a margin.  The loop that decodes by itself gives the tokens of its steps one by one, bit for bit."""
    from powerinfer_amd.model import Model
    hp = synth.hparams("llama-tiny", n_embd=d, n_head=heads, n_head_kv=kv_heads, n_rank=rank, n_ff=ff, n_vocab=2048, n_ctx=144, seed=6, pred_margin=True)
    model = synth.make_model(hp)
    rng = np.random.default_rng(d + heads + rank)
    a, b = Model(hp).load(model), Model(hp).load(model)
    for n in (0, 1, 60, 136):
        b.set_capture(False)
        if n:
            toks = rng.integers(0, hp.n_vocab, n).astype(np.int32)
            a.decode(toks, 0)
            b.decode(toks, 0)
        b.set_capture(True)
        for k in range(4):
            t = int(rng.integers(0, hp.n_vocab))
            _, got = a.decode([t], n + k)
            _, want = b.decode([t], n + k)
            assert np.abs(got - want).max() < 2e-3 * np.abs(want).max()
            assert np.array_equal(a.step_active(1), b.step_active(1))
        tok = a.decode([t], n + 3)[0]
        free = a.generate(2)[0]
        assert [a.decode([tok], n + 4)[0], a.decode([int(free[0])], n + 5)[0]] == [int(v) for v in free]
    a.close()
    b.close()
