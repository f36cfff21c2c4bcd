"""What the device learns of the sequences' cells, on the CPU (fake_hip): the triples (sequence, place, cell) of every launch that carries some are stored here, in
reverse, as the kernels promise no order, and have to leave the lists that follow from the positions."""
import fake_hip

DEVICE = """
import numpy as np
from lerasun_models import odd_config, tokens, weights
from powerinfer_amd import lerasun, lib as pl

class Start(C.Structure):                      # as PassStart of runtime.hpp begins
    _fields_ = [("src", C.c_void_p), ("dst", C.c_void_p), ("words", C.c_size_t), ("append", C.c_void_p), ("n", C.c_int), ("lists", C.c_void_p), ("ld", C.c_size_t)]

lists, sent = {}, []
def store(at, n):
    t = np.ctypeslib.as_array(C.cast(at, C.POINTER(C.c_int32)), (n, 3)).copy()
    assert len(set(map(tuple, t[:, :2].tolist()))) == n, "a place twice in one launch"
    sent.append(n)
    for q, place, cell in t[::-1].tolist():
        lists[q, place] = cell

@C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))
def on_launch(name, args):
    try:
        if b"pass_start_kernel" in name:
            p = C.cast(args[0], C.POINTER(Start))[0]
            if p.n:
                store(p.append, p.n)
        elif b"cells_append_args_kernel" in name:
            store(args[0], C.cast(args[1], C.POINTER(C.c_int))[0])
        elif b"cells_append_kernel" in name:
            store(C.cast(args[0], C.POINTER(C.c_void_p))[0], C.cast(args[1], C.POINTER(C.c_int))[0])
    except BaseException as e:
        sent.append(e)
F.fake_watch(on_launch)
def holds(q, cells):
    for e in sent:
        if isinstance(e, BaseException):
            raise e
    got = [lists.get((q, k)) for k in range(len(cells))]
    assert got == [int(c) for c in cells], (q, got, list(cells))
cfg = odd_config()
m = lerasun.build(cfg, weights(cfg, 17), compute=pl.F32, n_ctx=512)
m.kv_cells_init(512)
step = lambda pos, masks: m.kv_cells_step(tokens(cfg, len(pos), 1), pos, masks, [], want_logits=False)
"""


def test_positions_that_go_back_within_a_step():
    """The list is rebuilt when a token turns out not to be behind its sequence's last: what was said of it before has to go."""
    fake_hip.run(DEVICE + """
pos = list(range(20, 120)) + list(range(20))
step(pos, [1] * 120)                                    # cells 0 .. 119
holds(0, np.argsort(pos))
step([150, 130, 140], [1, 1, 1])
holds(0, list(np.argsort(pos)) + [121, 122, 120])
both = list(range(200, 260)) + list(range(160, 200))    # a second sequence shares what the first takes, its own start among them
step([5, 0] + both, [2, 2] + [3] * 100)                 # cells 123 and 124, then 125 ..
shared = list(125 + np.argsort(both))
holds(0, list(np.argsort(pos)) + [121, 122, 120] + shared)
holds(1, [124, 123] + shared)
""")
