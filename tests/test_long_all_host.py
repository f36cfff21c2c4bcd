"""What the host does about the number of listed neurons in the longest F16 chunks of large layers, on the CPU (fake_hip; test_gpu_long_all.py has these chunks on the GPU)."""
import fake_hip

CODE = """
import numpy as np
from powerinfer_amd import lib as pl, synth
from powerinfer_amd.model import Model
d, ff, rank = 2048, 24832, 256
hp = synth.hparams("llama-tiny", n_layer=3, n_embd=d, n_head=16, n_head_kv=16, n_ff=ff, n_rank=rank, n_vocab=64, n_ctx=2048, use_rates=False)
m = Model(hp)
z = lambda r, c: np.zeros((r, c), np.float16)
for k, a in (("tok_embd", z(64, d)), ("output", z(64, d)), ("output_norm", np.ones(d, np.float32))):
    m.set_tensor(-1, k, a)
big = z(ff, d)
for il in range(hp.n_layer):
    for k, a in (("attn_norm", np.ones(d, np.float32)), ("ffn_norm", np.ones(d, np.float32)), ("wq", z(d, d)), ("wk", z(d, d)), ("wv", z(d, d)), ("wo", z(d, d)), ("ffn_up", big), ("ffn_gate", big),
                 ("ffn_down_t", big), ("fc1", z(rank, d)), ("fc2", z(ff, rank))):
        m.set_tensor(il, k, a)
m.finalize()

class Ask(C.Structure):                          # HostAsk of runtime.hpp
    _fields_ = [("word", C.c_void_p), ("tag", C.c_uint32)]

say, asked = None, []
@C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))
def watch(name, args):
    if b"ffn_union_list_kernel" in name:
        told = C.cast(args[6], C.POINTER(Ask))[0]
        asked.append(bool(told.word))
        if told.word and say:
            C.cast(told.word, C.POINTER(C.c_uint32))[0] = told.tag | say
F.fake_watch(watch)

def go(n, number):
    global say
    say = number
    asked.clear()
    F.fake_clear_counts()
    m.decode(np.zeros(n, np.int32), 0)
    return list(asked), count("ffn_union_down"), count("transpose_f16"), F.fake_live()

FFN = hp.n_layer - 1                             # (of the last layer a chunk leaves its keys and values)
"""


def test_which_product_and_which_copy():
    fake_hip.run(CODE + """
a, down, copies, live = go(1792, ff)
assert a == [False] * FFN and down == FFN and copies == 0        # nobody asks
a, down, copies, live = go(2000, ff - 128)
assert a == [True] * FFN and down == FFN and copies == 0         # not all of them: the listed rows
F.fake_limit(0)                                                  # no room for a copy: the rows as stored
assert go(2000, ff) == ([True] * FFN, FFN, FFN * 0, live)
F.fake_limit(2 * d * ff + 4096)                                  # room for one
a, down, copies, now = go(2000, ff)
assert a == [True] * FFN and down == FFN - 1 and copies == 1 and now - live >= 2 * d * ff
F.fake_limit(C.c_size_t(-1).value)
a, down, copies, now = go(2000, ff)
assert a == [True] * FFN and down == 0 and copies == FFN - 1     # the other one's
assert go(2000, ff) == ([True] * FFN, 0, 0, now)                 # found
assert go(2000, ff - 128) == ([True] * FFN, FFN, 0, now)
m.close()
""")


def test_a_launch_that_does_not_answer():
    """An error and not a wait for ever, nor the number of the call before."""
    fake_hip.run(CODE + """
assert go(2000, ff)[1] == 0
try:
    go(2000, 0)
    raise SystemExit("no error")
except RuntimeError as e:
    assert "answer" in str(e), e
assert go(2000, ff)[1] == 0                                      # and the next one goes on
m.close()
""")
