"""Host set-up without enough memory: the entry points that build patterns and numberings on the host, on one thread or
several, return an error status; none ends the process. Each limit runs in a child process whose address space is capped
a little above what it already uses, so that the allocations fail one after the other (no GPU needed: a pattern that gets
through fails at its first device allocation)."""
import os
import resource
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import ctypes, resource, sys
import numpy as np
lib = ctypes.CDLL(sys.argv[1])
entry, extra = sys.argv[2], int(sys.argv[3])
def p(a): return a.ctypes.data_as(ctypes.c_void_p)
nv, nt = 6000000, 200000
rng = np.random.default_rng(0)
base = rng.integers(0, nv - 4, nt)
T = np.ascontiguousarray(base[:, None] + np.arange(4), np.int32)
X = rng.random((nv, 3)) if entry == "sk_part_order" else np.zeros((1, 3))
D = np.zeros((nt, 12))
order, n, ptr, out = np.empty(nv, np.int32), ctypes.c_int(), np.empty(257, np.int32), ctypes.c_void_p()
I64 = ctypes.c_int64
args = {"sk_mesh_create": (p(T), p(D), I64(nv), I64(nt), ctypes.byref(out)),
        "sk_sell_order": (p(T), I64(nv), I64(nt), p(order)),
        "sk_part_order": (p(X), p(T), I64(100000), I64(1000), 0, p(order), ctypes.byref(n), p(ptr))}[entry]
if entry == "sk_part_order":
    T[:1000] %= 100000
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + extra, resource.RLIM_INFINITY))
print("status", getattr(lib, entry)(*args), flush=True)
"""


# the mesh's vectors are 24 MB each (six million vertices), eight threads holding one or two of their own; the numberings'
# at most 24 MB and 0.4 MB
@pytest.mark.parametrize("entry,extra", [("sk_mesh_create", mb) for mb in (4, 60, 100, 140, 200, 300)] +
                         [("sk_sell_order", mb) for mb in (4, 40, 70)] + [("sk_part_order", 0)])
def test_out_of_host_memory_is_a_status(entry, extra):
    lib = os.path.join(ROOT, "simkit_amd", "libsimkit_amd.so")
    run = subprocess.run([sys.executable, "-c", CHILD, lib, entry, str(extra << 20)], capture_output=True, text=True,
                         timeout=100, preexec_fn=lambda: resource.setrlimit(resource.RLIMIT_CORE, (0, 0)))
    assert run.returncode == 0, (run.returncode, run.stderr[-400:])
    assert run.stdout.startswith("status"), run.stdout
    assert int(run.stdout.split()[1]) < 0, run.stdout
