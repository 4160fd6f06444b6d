"""COO entries in no order, sorted by the plan: forced on (small matrices) over row lengths around chunks and
column blocks, duplicates, rows without entries, the three element types, rows of every layout of the gather
kernels and the slices of K; the rule that turns it on; against the oracle.  All GPU.  Same bar as
test_gpu_parity.py."""
import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O
from test_gpu_row_lengths import _bits

pytestmark = pytest.mark.gpu
f32 = np.float32


def _entries(rng, M, N, lens):
    r = np.repeat(rng.permutation(M)[:len(lens)], lens)
    c = rng.integers(0, N, len(r))                       # some of them twice in a row
    p = rng.permutation(len(r))
    return r[p].astype(np.int32), c[p].astype(np.int32), rng.uniform(-1, 1, len(r)).astype(f32)


def _operands(rng, M, N, K, dtype):
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    if dtype == capi.BF16:
        A, B = capi.from_bf16(capi.to_bf16(A)), capi.from_bf16(capi.to_bf16(B))
    elif dtype == capi.F16:
        A, B = capi.from_f16(capi.to_f16(A)), capi.from_f16(capi.to_f16(B))
    return A, B


def _check(got, r, c, v, A, B, what):
    order = np.lexsort((c, r))
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=len(A)))]).astype(np.int32)
    ref = O.sddmm_csr(rowptr, c[order], v[order], A, B, threads=0)
    _, mag = O.sddmm_csr_f64(rowptr, c[order], v[order], A, B)
    ok, worst, i = O.check_values(got[order], ref, mag=mag)
    assert ok, "%s: entry %d got %r ref %r (%.2f x tolerance)" % (what, i, got[order][i], ref[i], worst)


PATTERNS = {
    "short": [1, 2, 3, 5, 8, 13, 21] * 40,
    "long": [1, 300, 257, 256, 63, 64, 65, 2000, 7] * 3,
    "one entry": [1],
    "two rows": [777, 1],
}


@pytest.mark.parametrize("K,dtype", [(1, capi.F32), (7, capi.F32), (32, capi.F32), (48, capi.F16), (75, capi.F32),
                                     (200, capi.BF16), (400, capi.F32), (601, capi.F32)])
@pytest.mark.parametrize("blocks", ["0", "1"])
def test_sorted_order(engine_factory, monkeypatch, K, dtype, blocks):
    monkeypatch.setenv("SDDMM_ORDER", "1")
    monkeypatch.setenv("SDDMM_COLUMN_BLOCKS", blocks)
    rng = np.random.default_rng(K)
    M, N = 400, 333
    A, B = _operands(rng, M, N, K, dtype)
    with engine_factory() as e:
        e.set_dense(_bits(A, dtype), _bits(B, dtype), dtype)
        for name, lens in PATTERNS.items():
            r, c, v = _entries(rng, M, N, lens)
            for slices in ("0", "1"):
                print("order", K, dtype, blocks, name, slices, flush=True)
                monkeypatch.setenv("SDDMM_SLICES", slices)
                e.set_coo(M, N, r, c, v)
                e.plan(capi.AUTO)
                e.run()
                st = e.stats()
                got = e.values()
                what = "%s K=%d slices=%s" % (name, K, slices)
                assert st.strategy_used == capi.FLAT, what
                size = 4 if dtype == capi.F32 else 2
                sliced, in_registers = slices == "1" and K * size > 128, K * size <= 2048
                variant = capi.FLAT_SLICES if sliced else 0
                if (np.diff(r) < 0).any() and (sliced or in_registers):
                    variant |= capi.FLAT_SORTED | (0 if sliced else capi.FLAT_BLOCKS)
                assert e.flat_variant() == variant, what
                assert st.kernels_launched == (2 if sliced else 1) + (1 if variant & capi.FLAT_SORTED else 0), what
                _check(got, r, c, v, A, B, what)
                if slices == "0":                        # the same arithmetic per entry as the plain kernel
                    e.set_coo(M, N, r, c, v)
                    e.plan(capi.FLAT)
                    e.run()
                    np.testing.assert_array_equal(e.values(), got)


def test_every_row_long(engine_factory, monkeypatch):
    """More column blocks of long rows than a scan in one workgroup takes, in a matrix of few rows."""
    monkeypatch.setenv("SDDMM_ORDER", "1")
    monkeypatch.setenv("SDDMM_COLUMN_BLOCKS", "1")
    rng = np.random.default_rng(5)
    M, N, K = 1100, 5000, 8
    A, B = _operands(rng, M, N, K, capi.F32)
    r, c, v = _entries(rng, M, N, [300] * M)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_coo(M, N, r, c, v)
        e.plan(capi.AUTO)
        e.run()
        assert e.stats().kernels_launched == 2
        _check(e.values(), r, c, v, A, B, "every row long")


def test_sorted_order_in_ranges_of_the_slice_workspace(engine_factory, monkeypatch):
    monkeypatch.setenv("SDDMM_ORDER", "1")
    monkeypatch.setenv("SDDMM_SLICES", "1")
    monkeypatch.setenv("SDDMM_SLICE_WORKSPACE", "1")     # the least: one wavefront's entries at a time
    rng = np.random.default_rng(3)
    A, B = _operands(rng, 90, 500, 80, capi.F32)
    r, c, v = _entries(rng, 90, 500, [30] * 41)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_coo(90, 500, r, c, v)
        e.plan(capi.AUTO)
        for _ in range(2):                               # and new values of S under the same plan
            e.run()
            _check(e.values(), r, c, v, A, B, "ranges")
            v = rng.uniform(-1, 1, len(r)).astype(f32)
            e.update_values(v)


def test_when_the_plan_sorts(engine_factory):
    """Shuffled entries over rows of 300 bytes are sorted (a second launch brings P back); entries grouped by
    column, few entries, short rows and FLAT by name are not."""
    rng = np.random.default_rng(9)
    M, N, K = 20000, 9000, 75
    lens = rng.integers(10, 60, 16000)
    r, c, v = _entries(rng, M, N, lens)
    A, B = _operands(rng, M, N, K, capi.F32)
    by_col = np.argsort(c, kind="stable")
    cases = [("shuffled", r, c, v, K, capi.AUTO, 2), ("by column", r[by_col], c[by_col], v[by_col], K, capi.AUTO, 1),
             ("few", r[:9999], c[:9999], v[:9999], K, capi.AUTO, 1), ("short rows", r, c, v, 32, capi.AUTO, 1),
             ("by name", r, c, v, K, capi.FLAT, 1)]
    with engine_factory() as e:
        for name, rr, cc, vv, k, strategy, launches in cases:
            print(name, flush=True)
            a, b = np.ascontiguousarray(A[:, :k]), np.ascontiguousarray(B[:, :k])
            e.set_dense(a, b)
            e.set_coo(M, N, rr, cc, vv)
            e.plan(strategy)
            e.run()
            st = e.stats()
            assert (st.strategy_used, st.kernels_launched) == (capi.FLAT, launches), name
            _check(e.values(), rr, cc, vv, a, b, name)


def test_sorted_by_64_bit_keys(engine_factory, monkeypatch):
    """2^28 rows and more: row and column block no longer fit 32 bits."""
    monkeypatch.setenv("SDDMM_ORDER", "1")
    rng = np.random.default_rng(28)
    M, N = (1 << 28) + 100, 50
    r = np.concatenate([rng.integers(0, M, 3000), np.arange(M - 60, M), [0, 0, 5], np.full(400, M - 7)])
    r = rng.permutation(r).astype(np.int32)
    c, v = rng.integers(0, N, len(r)).astype(np.int32), rng.uniform(-1, 1, len(r)).astype(f32)
    A, B = np.zeros((M, 1), f32), rng.uniform(-1, 1, (N, 1)).astype(f32)
    A[r, 0] = rng.uniform(-1, 1, len(r)).astype(f32)
    print("2^28 rows", flush=True)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_coo(M, N, r, c, v)
        e.plan(capi.AUTO)
        assert e.flat_variant() == capi.FLAT_SORTED | capi.FLAT_BLOCKS
        for _ in range(2):
            e.run()
            np.testing.assert_array_equal(e.values(), A[r, 0] * B[c, 0] * v)    # one product and its scaling: no sum
            e.plan(capi.AUTO)
