"""Rows of no whole number of 64-byte steps on the tile and panel kernels (RaggedRows): every length at which the kernels'
number of steps, the last step or the last unit changes, against the oracle and against the gather kernels."""
import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32


def _structured(seed, near_dense=1100):
    """Dense 16x16 tiles, a partly filled strip, 8-row panels (cut lists among them), near-dense rows between short ones;
    M and N are no multiples of 16."""
    rng = np.random.default_rng(seed)
    N = 611
    rows = []
    for _ in range(6):                                           # full and half-full tiles
        picks = rng.choice(N // 16, 9, replace=False)
        c = np.sort((picks[:, None] * 16 + np.arange(16)[None, :]).ravel())
        keep = rng.random((16, len(c))) < rng.choice([0.75, 1.0])
        rows += [c[k] for k in keep]
    rows += [np.arange(N - 40, N)] * 16                          # the last, narrower tile column
    for length in (17, 64, 65, 100, 610):                        # panels
        c = np.sort(rng.choice(N, length, replace=False))
        rows += [c] * 8
    for i in range(near_dense):                                  # near-dense rows in a window, short ones in between
        lo = int(rng.integers(0, N - 180))
        rows.append(lo + np.flatnonzero(rng.random(180) < 0.6))
        for _ in range(int(rng.integers(0, 3))):
            rows.append(np.sort(rng.choice(N, int(rng.integers(0, 20)), replace=False)))
    rows += [np.sort(rng.choice(N, 30, replace=False))] * 5      # the last rows are no whole strip
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    return len(rows), N, rowptr, col, rng.uniform(-1, 1, len(col)).astype(f32), rng


def _operands(rng, M, N, K, dtype):
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    if dtype == capi.F32:
        return A, B, A, B
    to, back = (capi.to_bf16, capi.from_bf16) if dtype == capi.BF16 else (capi.to_f16, capi.from_f16)
    Ab, Bb = to(A).reshape(M, K), to(B).reshape(N, K)
    return Ab, Bb, back(Ab).reshape(M, K), back(Bb).reshape(N, K)


def _run(e, M, N, rowptr, col, val, Ad, Bd, dtype, strategy=capi.AUTO):
    e.set_dense(Ad, Bd, dtype)
    e.set_csr(M, N, rowptr, col, val)                            # clears P
    e.plan(strategy)
    e.run()
    return e.values(), e.stats()


# lengths around every number of steps the kernels are built for, and around the last unit of a row
KS = [(K, capi.F32) for K in (9, 12, 13, 15, 17, 20, 31, 33, 47, 48, 49, 63, 65, 95, 97, 100, 127, 129, 160, 191, 193, 255)]
KS += [(K, d) for d in (capi.BF16, capi.F16) for K in (24, 40, 56, 72, 104, 136, 192, 264, 392, 504)]


@pytest.mark.parametrize("K,dtype", KS)
def test_ragged_rows(engine_factory, monkeypatch, K, dtype):
    M, N, rowptr, col, val, rng = _structured(K)
    Ad, Bd, A, B = _operands(rng, M, N, K, dtype)
    ref = O.sddmm_csr(rowptr, col, val, A, B)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    e = engine_factory()
    monkeypatch.setenv("SDDMM_RAGGED", "1")                      # whatever the number of entries
    got, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    assert st.mfma_tiles > 0 and st.panels >= 4
    assert st.nnz_mfma + st.nnz_panel + st.nnz_short + st.nnz_medium + st.nnz_long == len(col)
    ok, worst, i = O.check_values(got, ref, mag=mag)
    assert ok, (K, dtype, i, got[i], ref[i], worst)
    e.run()
    np.testing.assert_array_equal(e.values(), got)
    # tiles and rows in launches of their own; panel lists cut at other places
    monkeypatch.setenv("SDDMM_FUSE", "0")
    monkeypatch.setenv("SDDMM_PANEL_SEG", "67")
    again, st2 = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    assert st2.kernels_launched == 3
    ok, worst, i = O.check_values(again, ref, mag=mag)
    assert ok, (K, dtype, i, again[i], ref[i], worst)
    # by name the tile and panel kernels take whole steps only, and the gather kernels are still there
    for strategy in (capi.MFMA_TILE, capi.LDS_TILED):
        got, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype, strategy)
        assert st.mfma_tiles == 0 and st.panels == 0
        assert O.check_values(got, ref, mag=mag)[0]


@pytest.mark.parametrize("K,dtype", [(9, capi.F32), (31, capi.F32), (49, capi.F32), (100, capi.F32), (130, capi.F32),
                                     (24, capi.BF16), (136, capi.F16)])
def test_ragged_rows_keep_infinities_to_themselves(engine_factory, monkeypatch, K, dtype):
    """What a row holds at its end, where loads are clamped, and what lies behind it reach only the entries of that row:
    the same entries are finite as on the gather kernels."""
    M, N, rowptr, col, val, rng = _structured(1000 + K)
    _, _, A, B = _operands(rng, M, N, K, dtype)
    for k in (0, 3, K - 8 if K > 8 else 1, K - 4, K - 1):        # the start of a row, its last two units, its end
        A[int(rng.integers(0, M)), k] = np.inf
        B[int(rng.integers(0, N)), k] = np.nan
        B[int(rng.integers(0, N)), k] = -np.inf
    B[N - 1, K - 1] = np.inf
    A[M - 1, K - 1] = np.nan
    Ad, Bd = (A, B) if dtype == capi.F32 else [(capi.to_bf16 if dtype == capi.BF16 else capi.to_f16)(x).reshape(x.shape) for x in (A, B)]
    e = engine_factory()
    out = []
    for ragged in ("0", "1"):
        monkeypatch.setenv("SDDMM_RAGGED", ragged)
        got, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
        assert (st.mfma_tiles > 0 and st.panels > 0) == (ragged == "1")
        out.append(got)
    assert not np.isfinite(out[0]).all()
    np.testing.assert_array_equal(np.isfinite(out[1]), np.isfinite(out[0]))
    np.testing.assert_array_equal(np.isnan(out[1]), np.isnan(out[0]))


@pytest.mark.parametrize("K,dtype", KS)
def test_ragged_rows_tile_by_tile(engine_factory, monkeypatch, K, dtype):
    """The kernels of well-filled tiles, whatever the fill: tiles walked from their masks together with the rows, K split over the
    waves of a workgroup (from four steps on), a wavefront per window; non-finite values included."""
    M, N, rowptr, col, val, rng = _structured(2000 + K)
    Ad, Bd, A, B = _operands(rng, M, N, K, dtype)
    ref = O.sddmm_csr(rowptr, col, val, A, B)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    A, B = A.copy(), B.copy()
    for k in (0, K - 8 if K > 8 else 1, K - 4, K - 1):
        A[int(rng.integers(0, M)), k] = np.inf
        B[int(rng.integers(0, N)), k] = np.nan
    B[N - 1, K - 1] = -np.inf
    Ai, Bi = (A, B) if dtype == capi.F32 else [(capi.to_bf16 if dtype == capi.BF16 else capi.to_f16)(x).reshape(x.shape) for x in (A, B)]
    e = engine_factory()
    monkeypatch.setenv("SDDMM_RAGGED", "0")
    plain, _ = _run(e, M, N, rowptr, col, val, Ai, Bi, dtype)
    assert not np.isfinite(plain).all()
    monkeypatch.setenv("SDDMM_RAGGED", "1")
    monkeypatch.setenv("SDDMM_WINDOW_FILL", "0")                 # no windows
    for fuse, ksplit in (("1", "1"), ("0", "1"), ("0", "0")):
        monkeypatch.setenv("SDDMM_FUSE", fuse)
        monkeypatch.setenv("SDDMM_KSPLIT", ksplit)
        got, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
        assert st.mfma_tiles > 0 and st.kernels_launched == (2 if fuse == "1" else 3)
        ok, worst, i = O.check_values(got, ref, mag=mag)
        assert ok, (K, dtype, fuse, ksplit, i, got[i], ref[i], worst)
        got, _ = _run(e, M, N, rowptr, col, val, Ai, Bi, dtype)
        np.testing.assert_array_equal(np.isfinite(got), np.isfinite(plain))
        np.testing.assert_array_equal(np.isnan(got), np.isnan(plain))


LONG = [(K, capi.F32) for K in (257, 260, 300, 384, 511, 512, 516, 640, 1000, 1025)]
LONG += [(K, d) for d in (capi.BF16, capi.F16) for K in (520, 600, 768, 1024, 1032)]


@pytest.mark.parametrize("K,dtype", LONG)
def test_rows_beyond_1_kib(engine_factory, monkeypatch, K, dtype):
    """Tiles and panels of rows that the kernels take in several turns or launches; the rows that nobody owns stay with the
    gather kernels, and a matrix with many of them does as a whole."""
    M, N, rowptr, col, val, rng = _structured(K, near_dense=0)
    Ad, Bd, A, B = _operands(rng, M, N, K, dtype)
    ref = O.sddmm_csr(rowptr, col, val, A, B)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    monkeypatch.setenv("SDDMM_LONG_TILES", "1")
    e = engine_factory()
    got, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    assert st.mfma_tiles > 0 and st.panels >= 4 and st.strategy_used == capi.AUTO
    ok, worst, i = O.check_values(got, ref, mag=mag)
    assert ok, (K, dtype, i, got[i], ref[i], worst)
    e.run()                                                      # P is built up anew
    np.testing.assert_array_equal(e.values(), got)
    monkeypatch.setenv("SDDMM_PANEL_SEG", "67")
    got, _ = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    assert O.check_values(got, ref, mag=mag)[0]
    # non-finite values at the start and the end of a row, and of a turn
    for k in (0, 127, 128, 255, K - 1):
        if k < K:
            A[int(rng.integers(0, M)), k] = np.inf
            B[int(rng.integers(0, N)), k] = np.nan
    Ad, Bd = (A, B) if dtype == capi.F32 else [(capi.to_bf16 if dtype == capi.BF16 else capi.to_f16)(x).reshape(x.shape) for x in (A, B)]
    a, _ = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    monkeypatch.setenv("SDDMM_LONG_TILES", "0")
    b, st = _run(e, M, N, rowptr, col, val, Ad, Bd, dtype)
    assert st.mfma_tiles == 0 and st.panels == 0
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    np.testing.assert_array_equal(np.isfinite(a), np.isfinite(b))


def test_rows_beyond_1_kib_among_others(engine_factory, monkeypatch):
    M, N, rowptr, col, val, rng = _structured(5)                 # most entries in rows that nobody owns
    K = 300
    Ad, Bd, A, B = _operands(rng, M, N, K, capi.F32)
    monkeypatch.setenv("SDDMM_LONG_TILES", "1")
    got, st = _run(engine_factory(), M, N, rowptr, col, val, Ad, Bd, capi.F32)
    assert st.mfma_tiles == 0 and st.panels == 0
    ref = O.sddmm_csr(rowptr, col, val, A, B)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    assert O.check_values(got, ref, mag=mag)[0]


def test_ragged_rows_need_entries(engine_factory):
    """Few entries stay on the gather kernels, whatever their structure; rows beyond 1 KiB do too."""
    M, N, rowptr, col, val, rng = _structured(7, near_dense=20)
    for K in (20, 300):
        Ad, Bd, A, B = _operands(rng, M, N, K, capi.F32)
        got, st = _run(engine_factory(), M, N, rowptr, col, val, Ad, Bd, capi.F32)
        assert st.mfma_tiles == 0 and st.panels == 0
        ref = O.sddmm_csr(rowptr, col, val, A, B)
        _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
        assert O.check_values(got, ref, mag=mag)[0]
