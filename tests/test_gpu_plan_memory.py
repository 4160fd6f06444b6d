"""Arrays that a plan can do without, refused (SDDMM_SPARE_BYTES): the plan falls back to kernels that need none,
with the oracle's values.  All GPU.  Same bar as test_gpu_parity.py."""
import ctypes as C

import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32
M, N, NNZ = 900, 700, 20000


def _case(K, seed):
    rng = np.random.default_rng(seed)
    at = rng.choice(M * N, NNZ, replace=False)
    r, c = (at // N).astype(np.int32), (at % N).astype(np.int32)
    v = rng.uniform(-1, 1, NNZ).astype(f32)
    return r, c, v, rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)


def _check(got, r, c, v, A, B, what):
    rowptr, col, val = O.csr_from_triplets(M, r, c, v)
    order = np.lexsort((c, r))
    ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    ok, worst, i = O.check_values(got[order], ref, mag=mag)
    assert ok, "%s: entry %d got %r ref %r (%.2f x tolerance)" % (what, i, got[order][i], ref[i], worst)


# 20 000 entries: the sort's work arrays and the order take 0.32 MB each (and the sort some scratch memory), the slices
# of K = 601 1.6 MB
@pytest.mark.parametrize("K,limit,variant", [
    (601, None, capi.FLAT_SLICES | capi.FLAT_SORTED),
    (601, 1200000, 0),                                   # sorted, but no kernel without the slices takes the order
    (601, 0, 0),
    (100, None, capi.FLAT_BLOCKS | capi.FLAT_SORTED),
    (100, 100000, 0),
    (100, 0, 0),
])
def test_sorted_entries(engine_factory, monkeypatch, K, limit, variant):
    monkeypatch.setenv("SDDMM_ORDER", "1")
    if limit is not None:
        monkeypatch.setenv("SDDMM_SPARE_BYTES", str(limit))
    r, c, v, A, B = _case(K, K)
    print("sorted entries", K, limit, flush=True)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_coo(M, N, r, c, v)
        e.plan(capi.AUTO)
        assert e.flat_variant() == variant
        e.run()
        _check(e.values(), r, c, v, A, B, "K=%d limit=%s" % (K, limit))


@pytest.mark.parametrize("K,env,variant", [
    (300, {"SDDMM_SLICES": "1"}, capi.FLAT_SLICES),
    (601, {}, capi.FLAT_SLICES),
    (32, {"SDDMM_COLUMN_BLOCKS": "1", "SDDMM_SLICES": "0", "SDDMM_SEG": "64"}, capi.FLAT_BLOCKS),
    (32, {"SDDMM_FLAT_AVG": "0", "SDDMM_SLICES": "0"}, 0),           # entry list of the short rows
])
def test_csr(engine_factory, monkeypatch, K, env, variant):
    for name, value in dict(env, SDDMM_TILE_FILL="100000", SDDMM_UNION="0", SDDMM_GATHERED="0").items():
        monkeypatch.setenv(name, value)
    r, c, v, A, B = _case(K, K)
    c[:200] = np.arange(200) * 3                          # one long row
    r[:200] = 5
    keep = np.unique(r.astype(np.int64) * N + c, return_index=True)[1]
    r, c, v = r[keep], c[keep], v[keep]
    rowptr, col, val = O.csr_from_triplets(M, r, c, v)
    for limit in (None, 0):
        if limit is not None:
            monkeypatch.setenv("SDDMM_SPARE_BYTES", str(limit))
        print("csr", K, env, limit, flush=True)
        with engine_factory() as e:
            e.set_dense(A, B)
            e.set_csr(M, N, rowptr, col, val)
            e.plan(capi.AUTO)
            assert e.flat_variant() == (variant if limit is None else 0)
            e.run()
            _check(e.values(), r, c, v, A, B, "K=%d %s limit=%s" % (K, env, limit))


def test_the_work_arrays_of_the_sort_are_given_back(engine_factory):
    """A plan that sorts the entries keeps the sorted order, 16 bytes per entry, and not what the sort worked in."""
    rng = np.random.default_rng(17)
    rows, nnz, K = 40000, 3000000, 64
    r, c = rng.integers(0, rows, nnz).astype(np.int32), rng.integers(0, rows, nnz).astype(np.int32)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    with engine_factory() as e:
        e.set_dense(rng.uniform(-1, 1, (rows, K)).astype(f32), rng.uniform(-1, 1, (rows, K)).astype(f32))
        e.set_coo(rows, rows, r[:nnz // 2], c[:nnz // 2], np.ones(nnz // 2, f32))
        e.plan(capi.AUTO)                                 # what a process pays for once
        assert e.flat_variant() & capi.FLAT_SORTED
        e.set_coo(rows, rows, r, c, np.ones(nnz, f32))
        e.plan(capi.FLAT)
        before = free()
        e.plan(capi.AUTO)
        assert e.flat_variant() == capi.FLAT_SORTED | capi.FLAT_BLOCKS
        kept = before - free()
        print("kept", kept / nnz, "bytes per entry", flush=True)
        # 16 bytes and 0.3 for the work items; the arrays by rows and what the allocator rounds up to
        assert kept < 17 * nnz + (8 << 20)
        e.plan(capi.AUTO)                                 # planned again: the same
        assert before - free() < 17 * nnz + (8 << 20)
