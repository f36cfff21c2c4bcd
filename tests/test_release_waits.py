"""A release writes the L2 back (buffer_wbl2), and the count or flag behind it may only leave when that has ended: the generated code of every source that publishes to other workgroups or to the
host has a wait for it between the two."""
import concurrent.futures
import glob
import os
import re
import subprocess

import pytest

from powerinfer_amd import build

SOURCES = [f for f in sorted(glob.glob(os.path.join(os.path.dirname(build.__file__), "csrc", "*.hip")))
           if re.search(r"__ATOMIC_RELEASE|__ATOMIC_ACQ_REL|__threadfence|pi_release", open(f).read())]
# its sums pass the caches store by store, and nothing else is handed over
PAST_THE_CACHES = ("sum_norm_route_kernel",)


def unwaited(text):
    """(kernel, instruction) of every write-back that a store or an atomic follows without a wait, and how many write-backs there are."""
    name, pending, bad, n = "", False, [], 0
    for line in text.splitlines():
        label, code = re.match(r"(_Z\w+):", line), line.strip()
        if label:
            name, pending = label.group(1), False
        elif code.startswith("buffer_wbl2"):
            pending, n = True, n + 1
        elif code.startswith("s_waitcnt") and "vmcnt(0)" in code:
            pending = False
        elif pending and re.match(r"(global|flat|buffer)_(store|atomic)|s_endpgm|s_setpc", code):
            bad.append((name, code))
            pending = False
    return bad, n


def test_reader():
    assert unwaited("_Zk:\n buffer_wbl2 sc1\n global_store_dword v0, v1, s[0:1]\n") == ([("_Zk", "global_store_dword v0, v1, s[0:1]")], 1)
    assert unwaited("_Zk:\n buffer_wbl2 sc1\n s_waitcnt vmcnt(0)\n global_store_dword v0, v1, s[0:1]\n") == ([], 1)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_waits_behind_write_backs():
    def code(f):
        return subprocess.run([build.HIPCC, *build.FLAGS, "-x", "hip", "-S", "--cuda-device-only", f, "-o", "-"], check=True, stdout=subprocess.PIPE, text=True).stdout
    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        found = [unwaited(t) for t in pool.map(code, SOURCES)]
    bad = [b for f, _ in found for b in f if not any(k in b[0] for k in PAST_THE_CACHES)]
    assert sum(n for _, n in found) >= 10 and not bad, bad
