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


@pytest.mark.parametrize("name,hot", [("llama-tiny", 1.0), ("falcon-tiny", 1.0), ("llama-tiny", 0.6)])
def test_a_whole_piece_of_a_q4_prompt_goes_one_way(name, hot):
    """Q4_0: up to 16 tokens behind the first 512 leave these a chunk of their own, 17 make them a piece of a longer one: the same cells, bit for bit."""
    hp = synth.hparams(name, n_rank=256, n_ctx=700, seed=9, wtype=synth.Q4_0, hot_frac=hot)
    model = synth.make_model(hp)
    prompt = np.random.default_rng(4).integers(0, hp.n_vocab, 602).astype(np.int32)
    m, after = fresh(hp, model), {}
    for n in (513, 520, 529, 530, 602):                 # (the token that ends a prompt goes by itself)
        m.decode(prompt[:n], 0)
        after[n] = m.decode([5], 512)[1]
    m.close()
    assert all(np.array_equal(a, after[602]) for a in after.values()), {n: float(np.abs(a - after[602]).max()) for n, a in after.items()}


LONG = [("llama-tiny", synth.F16, 1.0, 1600, [1500]), ("falcon-tiny", synth.F16, 1.0, 2400, [2300]), ("llama-tiny", synth.F16, 1.0, 16384, [2300]),
        ("llama-tiny", synth.F16, 1.0, 2400, [1100, 1200]), ("llama-tiny", synth.F16, 0.6, 1300, [1200]),
        ("llama-tiny", synth.Q4_0, 1.0, 1300, [1200]), ("falcon-tiny", synth.Q4_0, 1.0, 2100, [600, 1400]), ("llama-tiny", synth.Q4_0, 0.6, 1300, [1200])]


def eval_behind(om, prompt, steps, cur=None):
    """Logits behind the prompt and of the steps on; the tokens of the steps: given, or greedy.  (logits, tokens)"""
    tok, lg = om.eval(prompt, 0)
    out, toks = [lg], [tok]
    for i in range(steps):
        tok, lg = om.eval([cur[i] if cur else toks[-1]], len(prompt) + i)
        out.append(lg)
        toks.append(tok)
    return out, toks


@pytest.mark.timeout(600)
@pytest.mark.parametrize("name,wtype,hot,n_ctx,parts", LONG)
def test_long_prompts_match_the_oracle(name, wtype, hot, n_ctx, parts):
    """Chunks of more than 600 tokens, a remainder behind 2048 of them, a second chunk behind cells of the first, a cache beyond what the chunk kernels
    hold, Q4_0 and split models: the logits behind the prompt and six steps on against the CPU path, every greedy token, on margin-protected
    models.  F16: within 1e-2.  Q4_0: within that or twice what the CPU path departs from itself when its norm weights move by one unit in
    the last place, either way (an activation rounded to eight bits the other way is a visible share of a dot product)."""
    import oracle_lib as ol
    hp = synth.hparams(name, n_rank=256, n_ctx=n_ctx, seed=5, pred_margin=True, head_pair=2048, wtype=wtype, hot_frac=hot)
    model = synth.make_model(hp)
    prompt = np.random.default_rng(8).integers(0, hp.n_vocab, sum(parts)).astype(np.int32)
    rel = lambda a, b: float(np.abs(a - b).max() / np.abs(b).max())  # noqa: E731
    om = ol.OracleModel(model)
    want, toks = eval_behind(om, [int(t) for t in prompt], 6)
    om.close()
    median = most = 1e-2
    for to in (0.0, 2.0) if wtype == synth.Q4_0 else ():
        moved = dict(model, layers=[dict(L, attn_norm=np.nextafter(L["attn_norm"], np.float32(to))) for L in model["layers"]])
        om = ol.OracleModel(moved)
        own = [rel(a, b) for a, b in zip(eval_behind(om, [int(t) for t in prompt], 6, toks)[0], want)]
        om.close()
        median, most = max(median, 2 * float(np.median(own))), max(most, 2 * max(own))
    m, at = fresh(hp, model), 0
    for n in parts:
        tok, lg = m.decode(prompt[at:at + n], at)
        at += n
    errs, got = [rel(lg, want[0])], [tok]
    for i in range(6):
        tok, lg = m.decode([toks[i]], at + i)
        errs.append(rel(lg, want[i + 1]))
        got.append(tok)
    m.close()
    print(name, wtype, hot, parts, f"median {np.median(errs):.4f} of {median:.4f}, most {max(errs):.4f} of {most:.4f}", flush=True)
    assert got == toks
    assert np.median(errs) <= median and max(errs) <= most, errs
