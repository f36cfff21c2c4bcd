"""Falcon's attention and sparse FFN in one launch (F16, 8192 columns), against the launches one by one that a capturing model takes."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(300)
@pytest.mark.parametrize("heads,kv_heads,rank,ff", [(128, 8, 1024, 32768), (128, 16, 512, 36992), (64, 64, 512, 32896), (64, 8, 1024, 32768)])
def test_decode_beside_the_ffn(heads, kv_heads, rank, ff):
    """Contexts whose cells a head takes whole and split, few and many cells; as many of the FFN's partial vectors as its sums request ahead, and more.  Both sides round q, k, v, the probabilities and h to fp16 at the same places and sum in fp32
    in another order, so that a value may round to the neighbouring fp16 number: up to 2^-11 of it, over two layers 2e-3 of the largest of 2048 logits.  Every decision of
    the predictor has a margin.  The loop that decodes by itself gives the tokens of its steps one by one, bit for bit."""
    from powerinfer_amd.model import Model
    hp = synth.hparams("falcon-40b", n_layer=2, n_head=heads, n_head_kv=kv_heads, n_rank=rank, n_ff=ff, n_vocab=2048, seed=5, pred_margin=True)
    model = synth.make_model(hp)
    rng = np.random.default_rng(heads + rank)
    for n_ctx, prompts in ((96, (0, 1, 90)), (1200, (0, 9, 1190))):
        hp["n_ctx"] = n_ctx
        a, b = Model(hp).load(model), Model(hp).load(model)
        for n in prompts:
            b.set_capture(False)
            if n:
                toks = rng.integers(0, hp.n_vocab, n).astype(np.int32)
                a.decode(toks, 0)
                b.decode(toks, 0)
            b.set_capture(True)
            for k in range(3):
                t = int(rng.integers(0, hp.n_vocab))
                _, got = a.decode([t], n + k)
                _, want = b.decode([t], n + k)
                assert np.abs(got - want).max() < 2e-3 * np.abs(want).max()
                assert np.array_equal(a.step_active(1), b.step_active(1))
            tok = a.decode([t], n + 2)[0]
            free = a.generate(2)[0]
            assert [a.decode([tok], n + 3)[0], a.decode([int(free[0])], n + 4)[0]] == [int(v) for v in free]
        a.close()
        b.close()
