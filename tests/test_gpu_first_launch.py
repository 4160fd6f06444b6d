"""The first launch of a process: the plan has loaded the device code, so the launch neither waits for it nor
allocates, and may be captured at once.  Every case is a process of its own.  All GPU."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = """
import ctypes as C, sys
import numpy as np
sys.path.insert(0, %r)
from dphpc_amd import capi, workloads as W
w = W.make(%%r, "small", K=32)
e = capi.Engine(0)
e.set_dense(w.A, w.B)
e.set_csr(w.M, w.N, w.rowptr, w.col, w.sval)
""" % ROOT

# the longest launch of these is 0.05 ms; loading a family of kernels takes 3 to 13 ms
TIMED = """
e.plan(%d)
e.run()
ms = e.stats().run_ms
print(capi.STRATEGY_NAMES[e.stats().strategy_used], "run_ms", ms, flush=True)
assert ms < 1.0, ms
"""

FUSED = """
e.plan(capi.AUTO)
e.run_fused(fetch=False)
ms = e.stats().run_ms
print("fused run_ms", ms, flush=True)
assert ms < 1.0, ms
"""

# capture straight after the plan (or the warm-up call of the entry point that allocates nothing), no launch before it
CAPTURE = """
h = C.CDLL("libamdhip64.so")
vp = C.c_void_p
def ok(rc): assert rc == 0, rc
h.hipMalloc.argtypes = [C.POINTER(vp), C.c_size_t]
h.hipMemcpy.argtypes = [vp, vp, C.c_size_t, C.c_int]
h.hipStreamBeginCapture.argtypes = [vp, C.c_int]
h.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
h.hipGraphInstantiate.argtypes = [C.POINTER(vp), vp, vp, vp, C.c_size_t]
h.hipGraphLaunch.argtypes = [vp, vp]
h.hipStreamSynchronize.argtypes = [vp]
h.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
stream, graph, gexec = vp(), vp(), vp()
ok(h.hipStreamCreate(C.byref(stream)))
def upload(a):
    p = vp()
    ok(h.hipMalloc(C.byref(p), a.nbytes))
    ok(h.hipMemcpy(p, a.ctypes.data_as(vp), a.nbytes, 1))
    return p
def free():
    f, t = C.c_size_t(), C.c_size_t()
    ok(h.hipMemGetInfo(C.byref(f), C.byref(t)))
    return f.value
noalloc = %r
L = capi.load_library()
if noalloc:
    dev = [upload(x) for x in (w.A, w.B, w.rowptr, w.col, w.sval)]
    dP = upload(np.zeros(w.nnz, np.float32))
    ok(L.sddmm_launch_noalloc(w.M, w.N, w.K, 0, None, None, dev[2], None, None, None, stream))
    launch = lambda: L.sddmm_launch_noalloc(w.M, w.N, w.K, w.nnz, *dev, dP, stream)
else:
    e.plan(capi.AUTO)
    e.set_stream(stream.value)
    launch = lambda: L.sddmm_launch(e.h)
before = free()
ok(h.hipStreamBeginCapture(stream, 0))
ok(launch())
ok(h.hipStreamEndCapture(stream, C.byref(graph)))
assert free() == before
ok(h.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0))
from oracle import oracle as O
ref = O.sddmm_csr(w.rowptr, w.col, w.sval, w.A, w.B)
_, mag = O.sddmm_csr_f64(w.rowptr, w.col, w.sval, w.A, w.B)
for replay in range(3):
    ok(h.hipGraphLaunch(gexec, stream))
    ok(h.hipStreamSynchronize(stream))
    got = np.empty(w.nnz, np.float32)
    if noalloc: ok(h.hipMemcpy(got.ctypes.data_as(vp), dP, got.nbytes, 2))
    else: got = e.values()
    good, worst, i = O.check_values(got, ref, mag=mag)
    assert good, (replay, i, worst)
    e.run() if not noalloc else ok(launch())          # the program's own eager work between the replays
    ok(h.hipStreamSynchronize(stream))
"""


def _child(text, workload):
    print(workload, flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", (HEAD % workload) + text], cwd=ROOT, capture_output=True, text=True, timeout=100)
    print(r.stdout[-2000:], flush=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]


@pytest.mark.parametrize("workload,strategy", [("power_law", 0), ("power_law", 2), ("power_law", 3), ("power_law", 6),
                                               ("mixed_density", 0), ("fem_banded", 0), ("dense_tiles", 5)])
def test_the_plan_loads_the_code_of_its_launches(workload, strategy):
    _child(TIMED % strategy, workload)


@pytest.mark.parametrize("workload", ["power_law", "fem_banded"])
def test_the_timed_part_of_a_fused_call_starts_with_its_code_loaded(workload):
    _child(FUSED, workload)


@pytest.mark.parametrize("noalloc", [False, True])
def test_capture_without_a_launch_before_it(noalloc):
    _child(CAPTURE % noalloc, "mixed_density" if not noalloc else "power_law")
