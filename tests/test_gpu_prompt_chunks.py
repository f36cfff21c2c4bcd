"""Prompts through chunks of up to 2048 tokens (pi_model_decode): the step buffers, where chunks end, and the logits behind them."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


def fresh(hp, model):
    from powerinfer_amd.model import Model
    return Model(hp).load(model)


@pytest.mark.parametrize("first,then", [(40, 1100), (600, 1500)])
def test_a_prompt_behind_one_with_another_attention(first, then, monkeypatch):
    """A model's first prompt runs with PI_ATTN_CHUNK=scalar (chunks of 512 tokens), the next one without it in longer chunks: its logits are a fresh
    model's, bit for bit."""
    hp = synth.hparams("llama-tiny", n_rank=256, n_ctx=1600, seed=7)
    model = synth.make_model(hp)
    rng = np.random.default_rng(3)
    a, b = (rng.integers(0, hp.n_vocab, n).astype(np.int32) for n in (first, then))
    m = fresh(hp, model)
    monkeypatch.setenv("PI_ATTN_CHUNK", "scalar")
    m.decode(a, 0)
    monkeypatch.delenv("PI_ATTN_CHUNK")
    _, got = m.decode(b, 0)
    m.close()
    f = fresh(hp, model)
    _, want = f.decode(b, 0)
    f.close()
    assert np.array_equal(got, want)
