"""Row lengths that are no power of two: the flat kernel in slices of K (rows of more than 128 bytes),
forced on wherever it can run, and the gather kernels on rows of no whole number of 16-byte units:
edges of lines, units, chunks and staged rows, against the oracle.  All GPU.

Same bar as test_gpu_parity.py.  B and A rows without entries hold NaN: every lane that
reads outside its entry's row (windows are moved down to lines) must leave the sum alone.
"""
import ctypes as C

import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O
from test_gpu_device_pointers import Hip

pytestmark = pytest.mark.gpu
f32 = np.float32


def _case(seed, M, N, K, dtype, nnz=None, density=0.3):
    rng = np.random.default_rng(seed)
    mask = rng.random((M, N)) < density
    mask[:, ::2] = False                                  # every other B row is nobody's
    mask[1::5] = False                                    # and every fifth A row
    r, c = np.nonzero(mask)
    if nnz is not None:
        assert len(r) >= nnz
        r, c = r[:nnz], c[:nnz]
    A = rng.uniform(-1, 1, (M, K)).astype(f32)
    B = rng.uniform(-1, 1, (N, K)).astype(f32)
    if dtype == capi.BF16:
        A, B = capi.from_bf16(capi.to_bf16(A)), capi.from_bf16(capi.to_bf16(B))
    elif dtype == capi.F16:
        A, B = capi.from_f16(capi.to_f16(A)), capi.from_f16(capi.to_f16(B))
    B[np.setdiff1d(np.arange(N), c)] = np.nan
    A[np.setdiff1d(np.arange(M), r)] = np.nan
    return r.astype(np.int32), c.astype(np.int32), rng.uniform(-1, 1, len(r)).astype(f32), A, B


def _bits(x, dtype):
    return x if dtype == capi.F32 else capi.to_bf16(x) if dtype == capi.BF16 else capi.to_f16(x)


def _check(got, r, c, v, A, B, what):
    M = A.shape[0]
    rowptr, col, val = O.csr_from_triplets(M, r, c, v)
    order = np.lexsort((c, r))
    ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    ok, worst, i = O.check_values(got[order], ref, mag=mag)
    assert ok, "%s: entry %d got %r ref %r (%.2f x tolerance)" % (what, i, got[order][i], ref[i], worst)


@pytest.fixture(autouse=True)
def _no_tiles(monkeypatch):
    """These patterns are dense enough for the matrix cores: keep every row on the gather kernels."""
    for name, value in (("SDDMM_TILE_FILL", "100000"), ("SDDMM_UNION", "0"), ("SDDMM_GATHERED", "0")):
        monkeypatch.setenv(name, value)


SHAPES = [(capi.F32, K) for K in (33, 36, 63, 64, 65, 94, 100, 127, 128, 131, 250, 513, 1000, 1001)] + \
         [(capi.BF16, K) for K in (72, 128, 136, 1032)] + [(capi.F16, K) for K in (72, 128, 2000)]


@pytest.mark.parametrize("dtype,K", SHAPES)
def test_slices_any_row_length(engine_factory, monkeypatch, dtype, K):
    monkeypatch.setenv("SDDMM_SLICES", "1")
    # rows of many entries (A staged in LDS), rows of one or two (A gathered), a bit of both
    for seed, M, N, density in ((1, 60, 150, 0.6), (2, 700, 61, 0.04), (3, 150, 90, 0.3)):
        r, c, v, A, B = _case(K + seed, M, N, K, dtype, density=density)
        print("slices", dtype, K, M, N, len(r), flush=True)
        rowptr, col, val = O.csr_from_triplets(M, r, c, v)
        with engine_factory() as e:
            e.set_dense(_bits(A, dtype), _bits(B, dtype), dtype)
            e.set_csr(M, N, rowptr, col, val)
            e.plan(capi.AUTO)
            e.run()
            assert e.stats().kernels_launched == 2
            _check(e.values(), r, c, v, A, B, "K=%d sorted" % K)
            perm = np.random.default_rng(seed).permutation(len(r))
            e.set_coo(M, N, r[perm], c[perm], v[perm])
            e.plan(capi.AUTO)
            e.run()
            assert e.stats().kernels_launched == 2
            _check(e.values(), r[perm], c[perm], v[perm], A, B, "K=%d unsorted" % K)


@pytest.mark.parametrize("nnz", [1, 63, 64, 65, 255, 256, 257, 1023, 1025, 2050])
def test_slices_entry_counts_and_ranges(engine_factory, monkeypatch, nnz):
    """Remainders of chunks, wavefronts and workgroups; and a workspace that holds a few hundred entries."""
    monkeypatch.setenv("SDDMM_SLICES", "1")
    K = 100
    r, c, v, A, B = _case(nnz, 90, 120, K, capi.F32, nnz=nnz, density=0.7)
    rowptr, col, val = O.csr_from_triplets(90, r, c, v)
    for workspace in (None, "1", "3000"):
        if workspace:
            monkeypatch.setenv("SDDMM_SLICE_WORKSPACE", workspace)
        print("slices nnz", nnz, workspace, flush=True)
        with engine_factory() as e:
            e.set_dense(A, B)
            e.set_csr(90, 120, rowptr, col, val)
            e.plan(capi.AUTO)
            e.run()
            _check(e.values(), r, c, v, A, B, "nnz=%d workspace=%s" % (nnz, workspace))


@pytest.mark.parametrize("K", [64, 100, 301])
def test_slices_follow_the_address_of_b(engine_factory, monkeypatch, K):
    """New A and B at another alignment keep the plan: the lines of a row follow the new address."""
    monkeypatch.setenv("SDDMM_SLICES", "1")
    r, c, v, A, B = _case(K, 80, 110, K, capi.F32)
    rowptr, col, val = O.csr_from_triplets(80, r, c, v)
    hip = Hip()
    e = engine_factory()                                   # creates the context (and selects the device) first
    try:
        for shift in (0, 4, 20, 28):                       # floats: 16-byte steps inside a 128-byte line
            lead = np.zeros(shift, f32)
            dA, dB = hip.upload(np.concatenate([lead, A.ravel()])), hip.upload(np.concatenate([lead, B.ravel()]))
            e._chk(e.L.sddmm_set_dense_device(e.h, 80, 110, K, dA.value + 4 * shift, dB.value + 4 * shift, capi.F32))
            if shift == 0:
                e.set_csr(80, 110, rowptr, col, val)
                e.plan(capi.AUTO)
            e.run()
            _check(e.values(), r, c, v, A, B, "K=%d shift=%d" % (K, shift))
    finally:
        e.close()                                          # the context goes first, the borrowed buffers after it
        hip.free_all()


def test_rows_beyond_the_register_layout_take_slices(engine_factory):
    """The rule itself: rows of more than 2 KB take slices under AUTO; FLAT by name stays one plain kernel."""
    r, c, v, A, B = _case(5, 70, 90, 515, capi.F32)
    rowptr, col, val = O.csr_from_triplets(70, r, c, v)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_csr(70, 90, rowptr, col, val)
        for strategy, launches in ((capi.AUTO, 2), (capi.FLAT, 1)):
            e.plan(strategy)
            e.run()
            assert e.stats().strategy_used == capi.FLAT and e.stats().kernels_launched == launches
            _check(e.values(), r, c, v, A, B, capi.STRATEGY_NAMES[strategy])


@pytest.mark.parametrize("K", [5, 6, 7, 9, 17, 30, 35, 62, 65, 97, 127, 129, 161, 193, 255, 257, 510, 511])
def test_rows_of_no_whole_number_of_units(engine_factory, monkeypatch, K):
    """K % 4 != 0 in the gather kernels: the last unit of a row ends with the row and overlaps the one before."""
    monkeypatch.setenv("SDDMM_SLICES", "0")
    for seed, M, N, density in ((1, 60, 150, 0.6), (2, 700, 61, 0.04)):
        r, c, v, A, B = _case(K + seed, M, N, K, capi.F32, density=density)
        print("unaligned", K, M, N, len(r), flush=True)
        rowptr, col, val = O.csr_from_triplets(M, r, c, v)
        with engine_factory() as e:
            e.set_dense(A, B)
            for strategy in (capi.FLAT, capi.ROW_WAVE, capi.SHORT_ROWS, capi.AUTO):
                e.set_csr(M, N, rowptr, col, val)         # clears P
                e.plan(strategy)
                e.run()
                _check(e.values(), r, c, v, A, B, "K=%d %s" % (K, capi.STRATEGY_NAMES[strategy]))


@pytest.mark.parametrize("slices", ["0", "1"])
@pytest.mark.parametrize("K", [131, 132])
def test_operand_beyond_4gib(engine_factory, monkeypatch, K, slices):
    """64-bit row offsets, with rows of no whole number of units and with slices of K."""
    monkeypatch.setenv("SDDMM_SLICES", slices)
    M, N = 40, (1 << 32) // (4 * K) + 100
    rng = np.random.default_rng(K)
    hot = np.unique(np.concatenate([np.arange(30), np.arange(N - 130, N), rng.integers(0, N, 100)]))
    B = rng.uniform(-1, 1, (len(hot), K)).astype(f32)
    A = rng.uniform(-1, 1, (M, K)).astype(f32)
    r, c = np.nonzero(rng.random((M, len(hot))) < 0.4)
    r, c = r.astype(np.int32), c.astype(np.int32)
    v = rng.uniform(-1, 1, len(r)).astype(f32)
    rowptr, col, val = O.csr_from_triplets(M, r, c, v)    # columns among the rows that are filled in
    print("wide", K, slices, "%.2f GiB" % (N * K * 4 / 2 ** 30), flush=True)
    hip = Hip()
    e = engine_factory()
    try:
        dA, dB = hip.upload(A), C.c_void_p()
        assert hip.h.hipMalloc(C.byref(dB), N * K * 4) == 0
        hip.live.append(dB)
        for i, n in enumerate(hot):
            assert hip.h.hipMemcpy(C.c_void_p(dB.value + int(n) * K * 4), B[i].ctypes.data_as(C.c_void_p), K * 4, 1) == 0
        e._chk(e.L.sddmm_set_dense_device(e.h, M, N, K, dA, dB, capi.F32))
        for strategy in (capi.AUTO, capi.FLAT, capi.ROW_WAVE):
            e.set_csr(M, N, rowptr, hot[col].astype(np.int32), val)
            e.plan(strategy)
            e.run()
            _check(e.values(), r, c, v, A, B, "K=%d %s" % (K, capi.STRATEGY_NAMES[strategy]))
    finally:
        e.close()
        hip.free_all()


@pytest.mark.parametrize("K,N,per_row,fewer,enough", [
    (256, 20000, 24, 11, 13),                             # 20 MB of B
    (256, 9000, 24, 19, 21),                              # 9 MB
    (100, 40000, 13, 11, 13),                             # 15 MB
    (256, 20000, 6, 23, 25),                              # rows of few entries
    (200, 20000, 6, 25, None),                            # and of 800 bytes
    (300, 9000, 6, None, 1),                              # rows beyond 1 KB: whatever the columns hold
    (256, 20000, 40, 11, 13),                             # against the row split: 20 MB of B
    (300, 20000, 40, 7, 9),                               # rows beyond 1 KB
    (256, 9000, 40, 47, 49),                              # 9 MB
])
def test_slices_where_the_columns_hold_enough_entries(engine_factory, monkeypatch, K, N, per_row, fewer, enough):
    """The rule by itself: a line of B has to be found in the L2 often enough."""
    rng = np.random.default_rng(K + N + per_row)
    for per_column, variant in ((fewer, 0), (enough, capi.FLAT_SLICES)):
        if per_column is None:
            continue
        M = N * per_column // per_row + 1
        print("reuse", K, N, per_row, per_column, flush=True)
        rowptr = (np.arange(M + 1) * per_row).astype(np.int32)
        col = rng.integers(0, N, M * per_row).astype(np.int32)
        val = np.ones(len(col), f32)
        A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
        with engine_factory() as e:
            e.set_dense(A, B)
            e.set_csr(M, N, rowptr, col, val)
            e.plan(capi.AUTO)
            assert e.flat_variant() == variant
            assert e.stats().strategy_used == (capi.FLAT if variant or per_row < 32 else capi.AUTO)
            e.run()
            ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
            ok, worst, i = O.check_values(e.values(), ref, mag=O.sddmm_csr_f64(rowptr, col, val, A, B)[1])
            assert ok, "%d per column: entry %d (%.2f x tolerance)" % (per_column, i, worst)
