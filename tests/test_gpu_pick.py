"""The greedy choice by several workgroups and the results it stores for the host: vocabularies of one workgroup and of many, at their edges and past the
pinned memory, ties in different workgroups, logits that are not numbers, single calls and replayed graphs in turn."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_vocab", [1, 6, 1024, 1027, 9001, 65536, 70001, 131100])
def test_choices(n_vocab):
    from powerinfer_amd.model import Model
    hp = synth.hparams("llama-tiny", n_vocab=n_vocab, n_ctx=64, seed=5, sparse_threshold=-1e30)
    made = synth.make_model(hp)
    out, rng = made["glob"]["output"], np.random.default_rng(n_vocab)
    # every 1000th row or so is one and the same, in most steps the largest or the smallest; one row is not a number
    same = np.unique(np.r_[n_vocab // 3, n_vocab - 1, rng.integers(0, n_vocab, n_vocab // 1000)])
    out[same] = rng.standard_normal(out.shape[1]).astype(np.float16)
    if n_vocab > 3:
        out[1] = np.nan
    gm = Model(hp).load(made)
    print(n_vocab, flush=True)
    tok, path = 0, []
    for pos in range(6):
        nxt, lg = gm.decode([tok], pos)
        assert lg.shape == (n_vocab,) and np.isnan(lg).sum() == (1 if n_vocab > 3 else 0)
        best = int(np.nanargmax(lg))
        assert nxt == best and (lg[same] == lg[same[0]]).all()
        assert gm.decode([tok], pos, want_logits=False)[0] == nxt
        path.append(nxt)
        tok = nxt
    for turn in range(2):                              # the same tokens from replays, with single calls between them
        gm.kv_clear()
        first, _ = gm.decode([0], 0, want_logits=False)
        rest, _ = gm.generate(5)
        assert [first] + rest.tolist() == path
        assert (gm.step_active(5) == hp.n_layer * hp.n_ff).all()
    gm.close()
