"""Device memory that is kept for the next pattern and the next context: results on blocks that held something else,
contexts on several threads, the bound, and that all of it can be given back.  All GPU.  Same bar as
test_gpu_parity.py."""
import ctypes as C
import threading

import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32


def _case(seed, K):
    rng = np.random.default_rng(seed)
    M, N = int(rng.integers(40, 3000)), int(rng.integers(64, 2000))
    lens = rng.integers(0, 40, M)
    lens[::max(1, M // 7)] = min(N, 300)
    lens[:16 * (seed % 3)] = N // 2                            # strips of well-filled tiles
    col = np.concatenate([np.sort(rng.choice(N, int(l), replace=False)) for l in lens]).astype(np.int32)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    val = rng.uniform(-1, 1, len(col)).astype(f32)
    return M, N, rowptr, col, val, A, B


def _check(got, M, N, rowptr, col, val, A, B, what):
    ref = O.sddmm_csr(rowptr, col, val, A, B)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    ok, worst, i = O.check_values(got, ref, mag=mag)
    assert ok, "%s: entry %d got %r ref %r (%.2f x tolerance)" % (what, i, got[i], ref[i], worst)


def _free():
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_patterns_in_turn(engine_factory):
    """One context, patterns of different sizes: blocks are used again with what an earlier pattern left in them."""
    L, p = capi.load_library(), C.c_void_p()
    at = []
    with engine_factory() as e:
        for seed in range(12):
            case = _case(seed, 32)
            print("pattern", seed, flush=True)
            e.set_dense(case[5], case[6])
            e.set_csr(*case[:5])
            e.plan(capi.AUTO)
            e.run()
            _check(e.values(), *case, "pattern %d" % seed)
            for _ in range(3):                                 # the results of one size: where those before them were
                e.set_csr(*case[:5])
                e._chk(L.sddmm_get_values_device(e.h, C.byref(p)))
                at.append(p.value)
    assert all(at) and len(set(at)) <= len(at) // 2, at


def test_contexts_on_several_threads():
    failures = []

    def work(t):
        try:
            for k in range(6):
                case = _case(100 + 10 * t + k, 64)
                got = capi.sddmm_csr(*case[2:], N=case[1])
                _check(got, *case, "thread %d call %d" % (t, k))
        except Exception as err:                               # noqa: BLE001
            failures.append(err)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures


def test_the_bound_and_the_way_back():
    L = capi.load_library()
    case = _case(1, 32)
    capi.sddmm_csr(*case[2:], N=case[1])                       # what a process pays for once
    assert L.sddmm_trim() == capi.OK
    before = _free()
    rng = np.random.default_rng(3)
    for k in range(10):                                        # 10 x 3 arrays of 20 .. 29 MB, of ten different sizes
        nnz = 5000000 + 250000 * k
        rowptr = np.linspace(0, nnz, 20001).astype(np.int32)
        A = np.ones((20000, 4), f32)
        got = capi.sddmm_csr(rowptr, rng.integers(0, 20000, nnz).astype(np.int32), np.ones(nnz, f32), A, A, strategy=capi.ROW_WAVE)
        assert (got == 4.0).all()
        kept = before - _free()
        print("kept after call", k, kept >> 20, "MiB", flush=True)
        assert 40 << 20 <= kept <= (128 << 20) + (8 << 20)     # the last call's arrays at least; and what the driver rounds up to
    assert L.sddmm_trim() == capi.OK
    assert before - _free() <= 8 << 20


def test_more_contexts_than_are_kept(engine_factory):
    """12 contexts open at once, all used, all closed, twice: 8 sets of streams and events are kept in between."""
    L = capi.load_library()
    assert L.sddmm_trim() == capi.OK
    streams = []
    for turn in range(2):
        engines = [engine_factory() for _ in range(12)]
        s = C.c_void_p()
        for k, e in enumerate(engines):
            case = _case(200 + k, 16)
            e.set_dense(case[5], case[6])
            e.set_csr(*case[:5])
            e.plan(capi.AUTO)
            e.run()
            _check(e.values(), *case, "context %d" % k)
            e._chk(L.sddmm_get_stream(e.h, C.byref(s)))
            streams.append(s.value)
        for e in engines:
            e.close()
    assert len(set(streams[:12])) == len(set(streams[12:])) == 12
    assert len(set(streams[:12]) & set(streams[12:])) >= 8
    assert L.sddmm_trim() == capi.OK
