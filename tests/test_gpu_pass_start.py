"""What a pass begins with in one launch or two: prompts at the edge between them, more new cells than one workgroup takes, more rotations than a launch holds,
sequences side by side, a call that is refused behind one that is not."""
import numpy as np
import pytest

from lerasun_models import tokens
from powerinfer_amd import lib as pl, serve
from pufivik_models import capped, config, talking
from test_gpu_pufivik import Oracle, check, model

pytestmark = pytest.mark.gpu


def turning_config():
    return config(96, 120, [(capped(2, 1, 24, 24, 9.0, base=300.0 + 50 * k) if k % 2 else talking(2, 1, 24, 24, rot=8 + 2 * (k % 5), base=900.0 + 10 * k)) for k in range(11)], groups=3, taps=3)


@pytest.mark.parametrize("compute", [pl.F32, pl.BF16], ids=["f32", "bf16"])
def test_prompts_and_rotations(compute):
    orc = Oracle(turning_config, compute)
    m = model(orc, compute, n_ctx=900)
    st = serve.Stepper(m, 900)
    for n, rid in ((127, "a"), (128, "b"), (129, "c"), (300, "d"), (1, "e")):
        toks = tokens(orc.cfg, n, n)
        print(n, flush=True)
        check(st.run([(rid, toks, list(range(n)))])[0], orc, toks, compute)
    both = [("f", tokens(orc.cfg, 70, 1), [69]), ("g", tokens(orc.cfg, 61, 2), [60])]
    got = st.run(both)[0]
    for row, (_, toks, places) in zip(got, both):
        check(row[None], orc, toks, compute, slice(places[0], places[0] + 1))
    for _ in range(2):
        with pytest.raises(pl.PiError):
            m.kv_cells_step([1] * 901, np.arange(901), [1 << 9] * 901, [900])
    more = tokens(orc.cfg, 61, 2) + [7]
    check(st.run([("g", [7], [0])])[0], orc, more, compute, slice(61, 62))
    m.close()
