"""Matrices whose work items would need 2^32 threads or more in one launch: the plan takes kernels that fit instead.
Made on the device (1.0e9 entries and more); the values of A and B make every sum exact.  All GPU."""
import ctypes as C

import pytest

from dphpc_amd import capi

pytestmark = pytest.mark.gpu


class _Borrowed:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 3}


def _device_array(torch, e, getter, shape):
    p = C.c_void_p()
    e._chk(getter(e.h, C.byref(p)))
    return torch.as_tensor(_Borrowed(p.value, shape), device="cuda")


def _matrix(torch, lens, N):
    """Row pointer and columns n % N of entry n: no two rows alike, no column twice in a row."""
    rowptr = torch.zeros(lens.numel() + 1, dtype=torch.int32, device="cuda")
    rowptr[1:] = torch.cumsum(lens, 0, dtype=torch.int64).int()
    nnz = int(lens.sum())
    assert nnz <= 2 ** 31 - 2 ** 16
    return rowptr, torch.arange(nnz, dtype=torch.int32, device="cuda").remainder_(N), nnz


def _operands(torch, M, N, K):
    """<A row, B row of column c> = c mod 128, exactly."""
    A = torch.zeros((M, K), device="cuda")
    A[:, 0] = 1.0
    B = torch.zeros((N, K), device="cuda")
    B[:, 0] = torch.arange(N, device="cuda").remainder(128).float()
    return A, B


def _check_p(P, col):
    step = 1 << 27
    for at in range(0, col.numel(), step):
        assert bool((P[at:at + step] == col[at:at + step].remainder(128).float()).all()), at


def test_column_blocks_of_too_many_long_rows(engine_factory, monkeypatch):
    """3.96 M rows of 257 entries would be 17 wavefronts each: beyond 2^26 wavefronts the plain kernel takes them."""
    import torch
    for name in ("SDDMM_UNION", "SDDMM_GATHERED"):                    # rows of neighbouring columns, all of them
        monkeypatch.setenv(name, "0")
    M, N, K, n_long = 34_500_000, 1_000_003, 4, 3_960_000
    lens = torch.ones(M, dtype=torch.int32, device="cuda")
    lens[8 * torch.arange(n_long, device="cuda")] = 257
    rowptr, col, nnz = _matrix(torch, lens, N)
    A, B = _operands(torch, M, N, K)
    S = torch.ones(nnz, device="cuda")
    torch.cuda.synchronize()
    print("long rows", M, nnz, flush=True)
    e = engine_factory()
    try:
        e._chk(e.L.sddmm_set_dense_device(e.h, M, N, K, A.data_ptr(), B.data_ptr(), capi.F32))
        e._chk(e.L.sddmm_set_csr_device(e.h, M, N, nnz, rowptr.data_ptr(), col.data_ptr(), S.data_ptr()))
        e.plan(capi.AUTO)
        assert e.stats().strategy_used == capi.FLAT and e.flat_variant() == 0
        e.run()
        _check_p(_device_array(torch, e, e.L.sddmm_get_values_device, (nnz,)), col)
    finally:
        e.close()
        del A, B, S, rowptr, col, lens
        torch.cuda.empty_cache()


def test_fused_call_with_too_many_rows_of_17_entries(engine_factory):
    """69 M rows of 17 entries among shorter ones would be work items of the fused call, a wavefront each: beyond
    2^26 of them they stay with the short rows."""
    import torch
    M, N, K = 161_000_000, 1_000_003, 4
    lens = torch.where(torch.arange(M, device="cuda").remainder_(7) < 3, 17, 1).int()
    assert int((lens == 17).sum()) > 1 << 26
    rowptr, col, nnz = _matrix(torch, lens, N)
    assert nnz < 8 * M                                                # mostly very short rows: 17 entries are long
    A, B = _operands(torch, M, N, K)
    S = torch.ones(nnz, device="cuda")
    squares = torch.zeros(nnz + 1, dtype=torch.int64, device="cuda")
    squares[1:] = torch.cumsum(col.remainder(128).long().square_(), 0)
    want = (squares[rowptr[1:].long()] - squares[rowptr[:-1].long()]).float()
    del squares, lens
    torch.cuda.synchronize()
    print("fused rows of 17", M, nnz, flush=True)
    e = engine_factory()
    try:
        e._chk(e.L.sddmm_set_dense_device(e.h, M, N, K, A.data_ptr(), B.data_ptr(), capi.F32))
        e._chk(e.L.sddmm_set_csr_device(e.h, M, N, nnz, rowptr.data_ptr(), col.data_ptr(), S.data_ptr()))
        e.run_fused(fetch=False)
        _check_p(_device_array(torch, e, e.L.sddmm_get_values_device, (nnz,)), col)
        out = _device_array(torch, e, e.L.sddmm_get_fused_device, (M, K))
        assert bool((out[:, 0] == want).all()) and not bool(out[:, 1:].any())
    finally:
        e.close()
        del A, B, S, rowptr, col, want
        torch.cuda.empty_cache()
