"""Results leave the device through pinned pieces of 512 KB (HostStage): logits whose size lies at the edges of a piece and of the ring of four."""
import numpy as np
import pytest

from powerinfer_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_vocab", [33, 8128, 8192, 9001, 32768, 40003])
def test_logits_arrive_whole(n_vocab):
    """16 equal sequences: equal rows, each the single sequence's logits to within the two kernels' orders of summation (products of 512
    fp16-rounded values: 1e-2 of the largest, the bound the batch tests use), and next tokens that are the rows' maxima."""
    from powerinfer_amd.model import Model
    hp = synth.hparams("llama-tiny", n_vocab=n_vocab, n_ctx=64, seed=11, sparse_threshold=-1e30)        # every neuron active: no mask to flip on a last place
    gm = Model(hp).load(synth.make_model(hp))
    gm.batch_init(16)
    for pos, tok in enumerate([3, n_vocab - 1, 7]):
        print(n_vocab, pos, flush=True)
        one, lg1 = gm.decode([tok], pos)
        nxt, lg = gm.batch_decode([tok] * 16, [pos] * 16)
        assert one == int(lg1.argmax()) and lg.shape == (16, n_vocab)
        assert np.isfinite(lg).all() and (lg == lg[0]).all() and (nxt == lg.argmax(1)).all()
        assert np.abs(lg[0] - lg1).max() <= 1e-2 * np.abs(lg1).max()
        none, nothing = gm.batch_decode([tok] * 16, [pos] * 16, want_logits=False)
        assert nothing is None and (none == nxt).all()
        again, lg2 = gm.decode([tok], pos, want_logits=False)
        assert again == one and lg2 is None
    gm.close()


def test_models_that_come_and_go():
    """A model's pinned memory passes to the next one: models made and closed in turn on four threads, every result as the first model's."""
    import threading

    from powerinfer_amd.model import Model
    hp = synth.hparams("llama-tiny", n_vocab=9001, n_ctx=64, seed=11, sparse_threshold=-1e30)
    weights, toks = synth.make_model(hp), [5, 8999, 17]

    def rows():
        gm = Model(hp).load(weights)
        out = [gm.decode([t], k)[1].copy() for k, t in enumerate(toks)]
        gm.close()
        return np.stack(out)

    want, got = rows(), []

    def work():
        for _ in range(3):
            got.append(rows())

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(len(got), flush=True)
    assert len(got) == 12 and all(np.array_equal(g, want) for g in got)


@pytest.mark.parametrize("n_vocab", [1000, 9001, 40003])
def test_no_step_gets_results_of_the_one_before(n_vocab):
    """Steps of two sets of tokens in turn, whose logits differ everywhere: every row is bit for bit what the same step gave when it was repeated, where results that are late are the same ones.
    16 rows are one piece of pinned memory, two, and five, which is more than the ring has; a single token's are stored by the launch that chooses the next one."""
    from powerinfer_amd.model import Model
    hp = synth.hparams("llama-tiny", n_vocab=n_vocab, n_ctx=64, seed=11, sparse_threshold=-1e30)
    gm = Model(hp).load(synth.make_model(hp))
    gm.batch_init(16)
    rng = np.random.default_rng(n_vocab)
    sets = rng.permutation(n_vocab)[:32].astype(np.int32).reshape(2, 16)
    where = np.zeros(16, np.int32)
    rows = [[(n.copy(), lg.copy()) for n, lg in (gm.batch_decode(s, where) for _ in range(3))][-1] for s in sets]
    ones = [[(n, lg.copy()) for n, lg in (gm.decode([s[0]], 0) for _ in range(3))][-1] for s in sets]
    assert (rows[0][1] != rows[1][1]).mean() > 0.99 and (ones[0][1] != ones[1][1]).mean() > 0.99
    for k in range(400):
        if k % 100 == 0:
            print(n_vocab, k, flush=True)
        i = k & 1
        nxt, lg = gm.batch_decode(sets[i], where)
        assert np.array_equal(lg, rows[i][1]) and np.array_equal(nxt, rows[i][0]), k
        one, lg = gm.decode([sets[i][0]], 0)
        assert one == ones[i][0] and np.array_equal(lg, ones[i][1]), k
    gm.close()
