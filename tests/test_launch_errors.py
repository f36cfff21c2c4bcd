"""A kernel launch that fails is the result of the call that made it, whichever of the call's launches it is.  On the CPU, over
entry points that run nothing and fail on request."""
import pytest

import fake_hip

# pointers nothing reads: multiples of 4096
CALLS = {
    "chunk": "L.pi_k_attn_chunk(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 64, None, None)",
    "chunk_one_token_per_workgroup": "L.pi_k_attn_chunk(P, 96, {T}, 1, 1, 32, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 32, None, None)",
    "chunk_long": "L.pi_k_attn_chunk_long(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 2, P, P, P, P, P, None, None)",
    "chunk_rows": "L.pi_k_attn_chunk_rows(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 64, None, None)",
}

RUN = """
from powerinfer_amd import lib
L, P, f = lib.load(), C.c_void_p(1 << 20), float
call = lambda: {call}
F.fake_fail_launch(-1)
assert call() == 0
n = F.fake_launches()
assert n >= 2, n
for k in range(n):
    F.fake_fail_launch(k)
    assert call() != 0, f"launch {{k}} of {{n}} failed and the call returned PI_OK"
"""


@pytest.mark.parametrize("T", [4, 40])
@pytest.mark.parametrize("name", sorted(CALLS))
def test_every_launch_of_a_chunks_attention(name, T):
    fake_hip.run(RUN.format(call=CALLS[name].format(T=T)))
