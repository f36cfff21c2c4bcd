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


def test_a_call_that_fails_loses_nothing():
    """Whichever launch of a step fails, one pass or several, and whatever refuses a call behind an edit of the cells: the next call's launches say what is missing."""
    fake_hip.run(DEVICE + """
L = pl.load()
def refused(f):
    try:
        f()
    except pl.PiError:
        return
    raise AssertionError("not refused")
for n in (40, 200):                                     # one launch that a pass begins with, two
    m.kv_cells_clear()
    lists.clear()
    F.fake_fail_launch(-1)
    step(range(n), [1] * n)
    launches = F.fake_launches()
    for k in range(launches):
        m.kv_cells_clear()
        lists.clear()
        F.fake_fail_launch(k)
        refused(lambda: step(range(n), [1] * n))
        F.fake_fail_launch(-1)
        step([n], [1])
        cells = [c for _, c in sorted((place, c) for (q, place), c in lists.items() if q == 0)]
        assert len(cells) == n + 1 and len(set(cells)) == n + 1, (n, k, len(cells))
m.close()

m = lerasun.build(cfg, weights(cfg, 17), compute=pl.F32, n_ctx=64)
lists.clear()
m.decode(list(range(1, 31)), 0)
kept = next(iter(lists))[0]                             # the model's own sequence
m.kv_seq_rm(10, 20)
m.kv_seq_shift(20, 30, -10)                             # the device's list still names the first thirty cells
refused(lambda: m.generate(60))                         # past the context, which is seen behind the rebuild of the list
m.decode([5], 20)
holds(kept, [*range(10), *range(20, 30), lists[kept, 20]])
m.close()
""")
