"""One token's attention launch also requests the weights behind it (load_ahead): the greedy run of whole models against the oracle where the
units do not divide evenly - heads that are no multiple of the eight XCDs, fewer units than XCDs or than
workgroups, and a width at which the 32 MB end inside wo."""
import pytest

from powerinfer_amd import synth
from test_gpu_model import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arch,wtype,over", [
    ("llama-tiny", synth.F16, dict(n_embd=192, n_head=3, n_head_kv=3, n_rank=32)),
    ("llama-tiny", synth.Q4_0, dict(n_embd=320, n_head=5, n_head_kv=5, n_rank=96)),
    ("falcon-tiny", synth.F16, dict(n_embd=320, n_head=5, n_head_kv=1, n_rank=32)),
    ("llama-tiny", synth.F16, dict(n_embd=4608, n_head=36, n_head_kv=36, n_rank=256, n_layer=1)),
])
def test_models_whose_units_do_not_divide_evenly(arch, wtype, over):
    print(arch, wtype, over, flush=True)
    run_case(synth.hparams(arch, wtype=wtype, n_ctx=64, seed=5, **over), n_prompt=4, n_gen=8)
