"""A kernel launch that fails is the result of the call that made it, whichever of the call's launches it is.  On the CPU: the HIP entry points of a
launch are replaced by ones that run nothing and fail on request."""
import os
import subprocess
import sys

import pytest

SHIM = r"""
#include <stddef.h>
static int n_launch, fail_at = -1, last;
typedef struct { unsigned x, y, z; } dim3_t;
void shim_reset(int k) { n_launch = 0; fail_at = k; last = 0; }
int shim_launches(void) { return n_launch; }
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void * st) { (void)g; (void)b; (void)sh; (void)st; return 0; }
int __hipPopCallConfiguration(dim3_t * g, dim3_t * b, size_t * sh, void ** st) { dim3_t one = {1, 1, 1}; *g = *b = one; *sh = 0; *st = 0; return 0; }
int hipLaunchKernel(const void * f, dim3_t g, dim3_t b, void ** a, size_t sh, void * st) {
    (void)f; (void)g; (void)b; (void)a; (void)sh; (void)st;
    return n_launch++ == fail_at ? (last = 1) : 0;
}
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipFuncSetAttribute(const void * f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipDeviceGetAttribute(int * v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetDevice(int * d) { *d = 0; return 0; }
"""

# pointers nothing reads: multiples of 4096
CALLS = {
    "chunk": "L.pi_k_attn_chunk(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 64, None, None)",
    "chunk_one_token_per_workgroup": "L.pi_k_attn_chunk(P, 96, {T}, 1, 1, 32, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 32, None, None)",
    "chunk_long": "L.pi_k_attn_chunk_long(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 2, P, P, P, P, P, None, None)",
    "chunk_rows": "L.pi_k_attn_chunk_rows(P, 192, {T}, 1, 1, 64, 0, f(0.9), f(1.0), P, 256, 0, P, P, P, P, 64, None, None)",
}

RUN = """
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L, P, f = C.CDLL(sys.argv[2]), C.c_void_p(1 << 20), C.c_float
call = lambda: {call}
shim.shim_reset(-1)
assert call() == 0
n = shim.shim_launches()
assert n >= 2, n
for k in range(n):
    shim.shim_reset(k)
    assert call() != 0, f"launch {{k}} of {{n}} failed and the call returned PI_OK"
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", "-o", str(d / "shim.so"), str(d / "shim.c")])
    return str(d / "shim.so")


@pytest.mark.parametrize("T", [4, 40])
@pytest.mark.parametrize("name", sorted(CALLS))
def test_every_launch_of_a_chunks_attention(name, T, shim):
    from powerinfer_amd import lib
    root = os.path.dirname(os.path.dirname(os.path.abspath(lib.__file__)))
    so = os.path.join(root, "powerinfer_amd", "libpowerinfer_hip.so")
    r = subprocess.run([sys.executable, "-c", RUN.format(call=CALLS[name].format(T=T)), shim, so], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-800:]
