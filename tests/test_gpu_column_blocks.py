"""The flat kernel with the long rows cut into column blocks, forced on (small matrices): row lengths around
the length that makes a row long, around whole pieces, long rows at either end and next to each other,
columns in one block only, unsorted rows; against the oracle.  All GPU.  Same bar as test_gpu_parity.py."""
import os

import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32


def _check(e, M, N, rowptr, col, val, A, B, dtype, what):
    e.set_dense(A if dtype == capi.F32 else capi.to_f16(A), B if dtype == capi.F32 else capi.to_f16(B), dtype)
    e.set_csr(M, N, rowptr, col, val)
    e.plan(capi.AUTO)
    assert e.stats().strategy_used == capi.FLAT, what
    longest, ts = int(np.diff(rowptr).max()), int(os.environ.get("SDDMM_TS", "24"))
    assert e.flat_variant() == (capi.FLAT_BLOCKS if longest > 256 and longest >= ts else 0), what
    e.run()
    ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    got = e.values()
    ok, worst, i = O.check_values(got, ref, mag=mag)
    assert ok, "%s: entry %d got %r ref %r (%.2f x tolerance)" % (what, i, got[i], ref[i], worst)
    # the same arithmetic per entry as the plain flat kernel
    e.set_csr(M, N, rowptr, col, val)
    e.plan(capi.FLAT)
    e.run()
    np.testing.assert_array_equal(e.values(), got)


def _matrix(rng, lens, N, kind="spread"):
    M = len(lens)
    cols = []
    for l in lens:
        if kind == "one block":
            c = np.sort(rng.choice(N // 16, size=min(int(l), N // 16), replace=False)) + N // 16 * 5
        else:
            c = np.sort(rng.choice(N, size=int(l), replace=False))
        if kind == "unsorted":
            c = rng.permutation(c)
        cols.append(c)
    rowptr = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    return M, rowptr, np.concatenate(cols).astype(np.int32), rng.uniform(-1, 1, rowptr[-1]).astype(f32)


@pytest.mark.parametrize("K,dtype", [(7, capi.F32), (32, capi.F32), (64, capi.F16), (100, capi.F32)])
@pytest.mark.parametrize("kind", ["spread", "one block", "unsorted"])
def test_column_blocks(engine_factory, monkeypatch, K, dtype, kind):
    monkeypatch.setenv("SDDMM_COLUMN_BLOCKS", "1")
    monkeypatch.setenv("SDDMM_SLICES", "0")
    N = 8 * 16 * 300 if kind == "one block" else 7001
    rng = np.random.default_rng(K)
    short = rng.integers(0, 9, 3000)
    patterns = {
        "edges": np.concatenate([[257, 256, 255], short[:1500], [512, 513, 4096, 1000], short[1500:], [300]]),
        "one long row": np.concatenate([short, [2000]]),
        "only at the start": np.concatenate([[258], short]),
        "scattered": np.concatenate([np.append(short[k * 60:(k + 1) * 60], 257 + 13 * k) for k in range(40)]),
    }
    A_all = rng.uniform(-1, 1, (4000, K)).astype(f32)
    B = rng.uniform(-1, 1, (N, K)).astype(f32)
    if dtype == capi.F16:
        A_all, B = capi.from_f16(capi.to_f16(A_all)), capi.from_f16(capi.to_f16(B))
    with engine_factory() as e:
        for name, lens in patterns.items():
            print("blocks", K, kind, name, flush=True)
            M, rowptr, col, val = _matrix(rng, lens, N, kind)
            _check(e, M, N, rowptr, col, val, A_all[:M], B, dtype, "%s %s K=%d" % (kind, name, K))
        # a pattern without a long row after one with: the plain kernel again
        M, rowptr, col, val = _matrix(rng, short, N, kind)
        _check(e, M, N, rowptr, col, val, A_all[:M], B, dtype, "no long row")


@pytest.mark.parametrize("kind", ["spread", "one block", "unsorted"])
@pytest.mark.parametrize("longest", [257, 1023, 1024, 2048, 4095, 4096, 9000])
def test_rows_around_the_numbers_of_blocks(engine_factory, monkeypatch, longest, kind):
    """8, 16, 32 and 64 blocks (from 1 024, 2 048 and 4 096 entries on), rows of every number in one matrix whose longest
    row sets the most there are; with the grid of a plan that the host has waited for and with that of one it has not."""
    monkeypatch.setenv("SDDMM_COLUMN_BLOCKS", "1")
    monkeypatch.setenv("SDDMM_SLICES", "0")
    N, K = 16 * 10000 if kind == "one block" else 12001, 8
    rng = np.random.default_rng(longest)
    edges = [257, 1023, 1024, 1025, 2047, 2048, 4095, 4096, 4097, 9000]
    lens = np.concatenate([[l for l in edges if l <= longest], rng.integers(0, 9, 4000), [l for l in edges if l <= longest], [3]])
    A = rng.uniform(-1, 1, (len(lens), K)).astype(f32)
    B = rng.uniform(-1, 1, (N, K)).astype(f32)
    with engine_factory() as e:
        print("numbers of blocks", longest, kind, flush=True)
        M, rowptr, col, val = _matrix(rng, lens, N, kind)
        _check(e, M, N, rowptr, col, val, A, B, capi.F32, "longest %d %s" % (longest, kind))
        want = e.values()
        e.set_csr(M, N, rowptr, col, val)
        e.plan(capi.AUTO)
        e.time_runs(0, 1, include_plan=True)
        assert e.flat_variant() == capi.FLAT_BLOCKS
        np.testing.assert_array_equal(e.values(), want)


@pytest.mark.parametrize("ts", [1, 257, 258, 600, 100000])
def test_rows_between_the_segment_length_and_the_short_row_limit(engine_factory, monkeypatch, ts):
    """SDDMM_TS above SDDMM_SEG: the rows in between are no long rows anywhere, neither in the count that sizes the
    list of the long rows nor in the list."""
    monkeypatch.setenv("SDDMM_COLUMN_BLOCKS", "1")
    monkeypatch.setenv("SDDMM_SLICES", "0")
    monkeypatch.setenv("SDDMM_TS", str(ts))
    N, K = 7001, 32
    rng = np.random.default_rng(ts)
    short = rng.integers(0, 9, 9000)                              # three blocks of the row scan
    lens = np.concatenate([[256, 257, 258], short[:2000], rng.integers(255, 602, 60), short[2000:], [599, 600, 601, 2500]])
    A = rng.uniform(-1, 1, (len(lens), K)).astype(f32)
    B = rng.uniform(-1, 1, (N, K)).astype(f32)
    with engine_factory() as e:
        print("between", ts, flush=True)
        M, rowptr, col, val = _matrix(rng, lens, N)
        e.set_dense(A, B)
        e.set_csr(M, N, rowptr, col, val)
        e.plan(capi.AUTO)
        assert e.flat_variant() == (capi.FLAT_BLOCKS if ts <= 2500 else 0)
        _check(e, M, N, rowptr, col, val, A, B, capi.F32, "ts=%d" % ts)


def test_when_the_plan_cuts_long_rows(engine_factory):
    """The rule by itself, on either side of each of its lines: 12 MB of B, 2^20 entries, a quarter of them in rows of
    more than 256."""
    rng = np.random.default_rng(11)
    N = 100000
    lens = np.concatenate([np.full(1400, 300), np.full(80000, 8)])
    rng.shuffle(lens)
    fewer, shorter = lens.copy(), lens.copy()
    fewer[np.flatnonzero(lens == 8)[:2000]] = 0                   # 1 044 000 entries
    shorter[np.flatnonzero(lens == 300)[:600]] = 256              # 240 000 of 1 033 600 in long rows ..
    shorter[np.flatnonzero(lens == 8)[:8000]] = 20                # .. of 1 129 600
    cases = [("all three", lens, 32, capi.FLAT_BLOCKS), ("11.2 MB", lens, 28, 0), ("few entries", fewer, 32, 0),
             ("few in long rows", shorter, 32, 0)]
    with engine_factory() as e:
        for name, lens_, K, variant in cases:
            print(name, flush=True)
            rowptr = np.concatenate([[0], np.cumsum(lens_)]).astype(np.int32)
            nnz, M = int(rowptr[-1]), len(lens_)
            assert (nnz >= 1 << 20) == (name != "few entries")
            col = rng.integers(0, N, nnz).astype(np.int32)
            A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
            e.set_dense(A, B)
            e.set_csr(M, N, rowptr, col, np.ones(nnz, f32))
            e.plan(capi.AUTO)
            assert (e.stats().strategy_used, e.flat_variant()) == (capi.FLAT, variant), name
            e.run()
            val = np.ones(nnz, f32)
            ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
            ok, worst, i = O.check_values(e.values(), ref, mag=O.sddmm_csr_f64(rowptr, col, val, A, B)[1])
            assert ok, "%s: entry %d (%.2f x tolerance)" % (name, i, worst)
