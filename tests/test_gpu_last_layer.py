"""The last layer of prompts: sparse models keep only its keys and values for the tokens of a chunk, models described layer by layer go on behind its
attention with the tokens whose logits are wanted."""
import numpy as np
import pytest

import fikevik_models
import lerasun_models
import pibalorn_models
import pufivik_models
from lerasun_models import row_errors, tokens
from powerinfer_amd import fikevik, lerasun, pibalorn, pufivik, synth

pytestmark = pytest.mark.gpu
FAMILIES = {"lerasun": (lerasun, lerasun_models), "pibalorn": (pibalorn, pibalorn_models), "fikevik": (fikevik, fikevik_models), "pufivik": (pufivik, pufivik_models)}


@pytest.mark.parametrize("name,layers,hot,ff", [("llama-tiny", 1, 1.0, 8192), ("llama-tiny", 3, 1.0, 8192), ("falcon-tiny", 1, 1.0, 8192), ("falcon-tiny", 2, 1.0, 8192), ("llama-tiny", 2, 0.6, 8192),
                                                ("llama-tiny", 2, 1.0, 4096), ("llama-tiny", 3, 1.0, 8448), ("falcon-tiny", 2, 1.0, 8448)])
@pytest.mark.parametrize("n", [3, 17, 18, 34, 131, 530])
def test_a_step_behind_a_prompt(name, layers, hot, ff, n):
    """Logits of the step behind a prompt, whose cells a chunk wrote, against those behind the same tokens one by one: both are sums of the same fp16
    products in fp32, 1e-2 as for the CPU path."""
    from powerinfer_amd.model import Model
    hp = synth.hparams(name, n_layer=layers, n_ff=ff, n_rank=256, n_ctx=600, seed=13, pred_margin=True, hot_frac=hot)
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


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("make", ["even_config", "odd_config"])
@pytest.mark.parametrize("n,want", [(17, [16]), (17, []), (40, [39, 3, 3]), (150, list(range(134, 150))), (150, list(range(133, 150))), (150, [])])
def test_wanted_rows(family, make, n, want):
    """One, none, some (out of order, twice), as many as a step holds and one more: logits against a pass that keeps every token's stream (the rows of
    the last layer are then products of the same bf16 values in another order, with the experts' sum rounded to bf16 on the way: 2^-8 of
    a row, times four), and the step behind, whose cells and states are the same, bit for bit."""
    lib, mod = FAMILIES[family]
    cfg = getattr(mod, make)()
    toks, out = tokens(cfg, n + 1, n), []
    w = mod.weights(cfg, 17)
    for keep in (True, False):
        m = lib.build(cfg, w, n_ctx=512)
        m.kv_cells_init(512)
        m.set_capture(keep)
        lg = m.kv_cells_step(toks[:n], range(n), [1] * n, want)[1]
        m.set_capture(False)
        out.append((lg, m.kv_cells_step(toks[n:], [n], [1], [0])[1]))
        m.close()
    (full, after), (got, then) = out
    assert np.array_equal(after, then)
    assert len(want) == 0 or (full.shape == got.shape == (len(want), full.shape[1]) and row_errors(got, full).max() < 2 ** -6)


@pytest.mark.parametrize("want", [[29], [69, 29, 0], list(range(54, 70)), []])
def test_wanted_rows_of_a_layer_without_cells(want):
    """Latent attention whose last layer reads the cells of the one before: two sequences' tokens in one pass, wanted rows of one and both (out of order),
    as many as a step holds, none.  The attention of these is the latent form instead of the expanded one, so against the CPU path, as
    test_gpu_lerasun.py has it."""
    import plain_latent
    import test_gpu_lerasun as lt
    cfg = lerasun_models.config(96, 101, [lerasun_models.layer(4, 16, 8, 24, 40), lerasun_models.layer(4, 16, 8, 24, 40, kv_from=0, moe=(6, 2, 3, 2, 24))])
    w = lerasun_models.weights(cfg, 17)
    a, b = tokens(cfg, 30, 1), tokens(cfg, 40, 2)
    m = lerasun.build(cfg, w, n_ctx=512)
    m.kv_cells_init(512)
    got = m.kv_cells_step(a + b, list(range(30)) + list(range(40)), [1] * 30 + [2] * 40, want)[1]
    after = m.kv_cells_step([5, 6], [30, 40], [1, 2], [0, 1])[1]
    m.close()
    runs = []
    for toks in (a + [5], b + [6]):
        p = plain_latent.PlainModel(cfg, w)
        lg = p.feed(toks)
        runs.append(lt.Logits(lg, np.asarray(p.margins)))
    full = lt.Logits(np.concatenate([np.asarray(runs[0])[:30], np.asarray(runs[1])[:40]]), np.concatenate([runs[0].margins[:30], runs[1].margins[:40]]))
    if want:
        lt.check(got, full[want], lt.pl.BF16)
    lt.check(after, lt.Logits(np.stack([np.asarray(r)[-1] for r in runs]), np.array([r.margins[-1] for r in runs])), lt.pl.BF16)
