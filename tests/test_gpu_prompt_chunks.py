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


@pytest.mark.parametrize("name,hot", [("llama-tiny", 1.0), ("falcon-tiny", 1.0), ("llama-tiny", 0.6)])
def test_cells_of_a_q4_prompt_do_not_depend_on_what_follows(name, hot):
    """Q4_0: the first 512 tokens leave the same cells behind, bit for bit, whether 90 or 1500 tokens come after them: products and attention
    keep one order of sums, so that no activation is rounded to eight bits the other way because the prompt is longer."""
    hp = synth.hparams(name, n_rank=256, n_ctx=2100, seed=9, wtype=synth.Q4_0, hot_frac=hot)
    model = synth.make_model(hp)
    rng = np.random.default_rng(4)
    prompt = rng.integers(0, hp.n_vocab, 2048).astype(np.int32)
    m, after = fresh(hp, model), {}
    for n in (602, 1001, 1030, 1100, 1541, 2048):
        m.decode(prompt[:n], 0)
        after[n] = m.decode([5], 512)[1]
    m.close()
    assert all(np.array_equal(a, after[602]) for a in after.values()), {n: float(np.abs(a - after[602]).max()) for n, a in after.items()}
