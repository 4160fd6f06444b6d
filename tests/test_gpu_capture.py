"""Work of other contexts while a stream is captured: patterns replaced, contexts created and destroyed.  In relaxed mode
and, from another thread, in thread-local mode none of that may break the capture.  All GPU.  Same bar as
test_gpu_parity.py."""
import ctypes as C
import threading

import numpy as np
import pytest

from dphpc_amd import capi
from test_gpu_device_pool import _case, _check

pytestmark = pytest.mark.gpu
THREAD_LOCAL, RELAXED = 1, 2


@pytest.mark.parametrize("mode", [THREAD_LOCAL, RELAXED])
@pytest.mark.parametrize("what", ["replace", "create", "destroy"])
def test_other_contexts_during_a_capture(engine_factory, mode, what):
    hip = C.CDLL("libamdhip64.so")
    stream, graph, executable = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    case, other = _case(300, 32), _case(301, 32)
    a, b = engine_factory(), engine_factory()
    for e, c in ((a, case), (b, other)):
        e.set_dense(*c[5:])
        e.set_csr(*c[:5])
        e.plan(capi.AUTO)
        e.run()
    a.set_stream(stream.value)
    a.launch()
    a.synchronize()
    failures = []

    def work():
        try:
            for k in range(3):
                c = _case(310 + k, 32)
                if what == "replace":
                    b.set_dense(*c[5:])
                    b.set_csr(*c[:5])
                    b.plan(capi.AUTO)
                    b.run()
                    _check(b.values(), *c, "replaced %d" % k)
                elif what == "create":
                    _check(capi.sddmm_csr(*c[2:], N=c[1]), *c, "created %d" % k)
            if what == "destroy":
                b.close()
        except Exception as err:                               # noqa: BLE001
            failures.append(err)

    assert hip.hipStreamBeginCapture(stream, mode) == 0
    a.launch()
    if mode == RELAXED:
        work()
    else:
        t = threading.Thread(target=work)
        t.start()
        t.join()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert not failures, failures
    assert hip.hipGraphInstantiate(C.byref(executable), graph, None, None, C.c_size_t(0)) == 0
    for k in range(3):
        a.update_values(case[4] * np.float32(2 ** k))
        assert hip.hipGraphLaunch(executable, stream) == 0
        a.synchronize()
        _check(a.values(), *case[:4], case[4] * np.float32(2 ** k), *case[5:], "replay %d" % k)
    assert hip.hipGraphExecDestroy(executable) == 0 and hip.hipGraphDestroy(graph) == 0
    a.close()
    assert hip.hipStreamDestroy(stream) == 0
