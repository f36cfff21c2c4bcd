"""Step buffers of long prompts, on the CPU (fake_hip): how much memory a model takes for the prompts it has seen, what it does where that much is
not to be had, and which kernels its layers go through."""
import fake_hip

MODEL = """
import numpy as np
from powerinfer_amd import lib as pl, synth
from powerinfer_amd.model import KIND, Model

def made(**kw):
    hp = synth.hparams("llama-tiny", n_rank=256, n_ctx=2100, seed=9, use_rates=False, **kw)
    return Model(hp).load(synth.make_model(hp)), hp

def prompt(m, n):
    F.fake_clear_counts()
    m.decode(np.zeros(n, np.int32), 0)
    return F.fake_live()
"""


def test_buffers_follow_the_prompts():
    """512 tokens first, twice and four times that when longer prompts come, nothing back and forth.  A resident F16 model has no up and gate products."""
    fake_hip.run(MODEL + """
m, hp = made()
a, b, c, d, e = (prompt(m, n) for n in (20, 500, 700, 1500, 2040))
assert a == b < c < d == e == prompt(m, 30), (a, b, c, d, e)
token = (c - b) / 512
assert abs((d - c) / 1024 - token) < 0.05 * token, (d - c, c - b)
need = 4 * (6 * hp.n_embd + 3 * hp.n_embd + hp.n_rank + hp.n_ff) + 2 * (4 * hp.n_embd + hp.n_rank + hp.n_ff)
assert need <= token < need + 1024, (token, need)
q, _ = made(wtype=synth.Q4_0)
a, b = prompt(q, 700), prompt(q, 1500)
assert (b - a) / 1024 >= need + 8 * hp.n_ff
m.close(); q.close()
""")


def test_without_memory_for_long_chunks_a_prompt_goes_by_512():
    fake_hip.run(MODEL + """
m, hp = made()
prompt(m, 20)
at_512 = F.fake_live()
prompt(m, 2040)
assert count("attn_chunk_rows") == hp.n_layer - 1               # (of the last layer a chunk leaves its keys and values)
at_2048 = F.fake_live()
n, hp = made()
prompt(n, 20)
F.fake_limit((at_2048 - at_512) // 2)
prompt(n, 2040)
assert count("attn_chunk_rows") == 4 * (hp.n_layer - 1), count("attn_chunk_rows")
F.fake_limit(C.c_size_t(-1).value)
prompt(n, 2040)                          # memory is there again
assert count("attn_chunk_rows") == hp.n_layer - 1
""")


def test_matrices_off_16_bytes_go_through_the_library():
    """Device tensors that start on 8 bytes: gate and up are products of the library, as they were before one kernel took both."""
    fake_hip.run(MODEL + """
for off in (0, 8):
    hp = synth.hparams("llama-tiny", n_rank=256, n_ctx=600, seed=9, use_rates=False)
    model, m = synth.make_model(hp), Model(hp)
    for k, a in model["glob"].items():
        m.set_tensor(-1, k, a)
    L = pl.load()
    for il, layer in enumerate(model["layers"]):
        for k, a in layer.items():
            if k in KIND and a is not None and k != "ffn_up":
                m.set_tensor(il, k, a)
        up = layer["ffn_up"]
        p = L.pi_malloc(up.nbytes + 16)
        m.set_tensor_device(il, "ffn_up", p + off, pl.F16, up.shape[1], up.shape[0])
    m.finalize()
    prompt(m, 200)
    assert (count("ffn_wide"), count("ffn_h_f16")) == ((hp.n_layer - 1, 0) if off == 0 else (0, hp.n_layer - 1)), off
    m.close()
""")


def test_chunks_whose_predictors_leave_bits():
    """Longer than one token tile; shorter ones, for which its tiles are too few, take the library's product and logits."""
    fake_hip.run(MODEL + """
m, hp = made()
for n, bits in ((30, 0), (129, 0), (130, 1), (600, 1)):
    prompt(m, n)
    assert (count("mask_wide") > 0) == bits and count("ffn_wide") > 0, n
m.close()
""")


def test_dense_feed_forwards_in_one_product():
    """From 1400 tokens on, where the rows of gate and up come in tiles of 128: gate, up and GLU are one product a layer (test_gpu_glu_in_one.py has
    these passes on the GPU).  Padded ones and shorter passes go apart."""
    fake_hip.run("""
import fikevik_models as fm
from lerasun_models import tokens
from powerinfer_amd import fikevik
for ff, whole in ((128, 1), (192, 0), (256, 1), (320, 0), (384, 1)):
    cfg = fm.config(256, 200, [fm.gla(2, 64, 64, mlp=fm.dense(ff)), fm.gla(4, 32, 64, mlp=fm.dense(ff))])
    m = fikevik.build(cfg, fm.weights(cfg, 5), n_ctx=2048, max_batch=2048)
    m.kv_cells_init(2048)
    for n in (1399, 1400, 1537):
        F.fake_clear_counts()
        m.kv_cells_step(tokens(cfg, n, 3), range(n), [1] * n, list(range(17)))
        assert count("group_wide") == (2 if whole and n >= 1400 else 0), (ff, n)
        m.kv_cells_clear()
    m.close()
""")
