"""Who owns a row where the rules of a plan meet: strips that are two panels, panel lists cut for the chip's wavefronts,
gathered pairs wider than the masks in LDS, classifiers of more rows than one pass, columns too far apart for ragged tiles."""
import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32


def _csr(rows):
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return rowptr, np.concatenate(rows).astype(np.int32)


def _check(engine_factory, rows, N, K, rng, dtype=capi.F32, coo=False, **counts):
    M = len(rows)
    rowptr, col = _csr(rows)
    val = rng.uniform(-1, 1, len(col)).astype(f32)
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    e = engine_factory()
    if dtype == capi.BF16:
        Ab, Bb = capi.to_bf16(A).reshape(M, K), capi.to_bf16(B).reshape(N, K)
        A, B = capi.from_bf16(Ab).reshape(M, K), capi.from_bf16(Bb).reshape(N, K)
        e.set_dense(Ab, Bb, dtype)
    else:
        e.set_dense(A, B)
    if coo:
        e.set_coo(M, N, np.repeat(np.arange(M, dtype=np.int32), np.diff(rowptr)), col, val)
    else:
        e.set_csr(M, N, rowptr, col, val)
    e.plan(capi.AUTO)
    st = e.stats()
    e.run()
    ref = O.sddmm_csr(rowptr, col, val, A, B, threads=0)
    _, mag = O.sddmm_csr_f64(rowptr, col, val, A, B)
    ok, worst, i = O.check_values(e.values(), ref, mag=mag)
    assert ok, (i, worst)
    assert st.nnz_mfma + st.nnz_panel + st.nnz_short + st.nnz_medium + st.nnz_long == len(col)
    for name, want in counts.items():
        assert getattr(st, name) == want, (name, getattr(st, name), want)
    e.close()
    return st


@pytest.mark.parametrize("K", [16, 32, 100, 256])
@pytest.mark.parametrize("full,loose,panels", [(9, 0, False), (0, 9, True), (7, 2, False), (1, 8, True), (1, 0, False),
                                               (0, 1, True)])
def test_strips_of_two_panels_go_one_way(engine_factory, monkeypatch, K, full, loose, panels):
    """full strips fill 80 % of their tiles, loose ones 49 %: tiles or panels, whichever suits the average, never both."""
    monkeypatch.setenv("SDDMM_RAGGED", "1")
    rng = np.random.default_rng(100 * full + loose)
    N, rows = 640, []
    for k in rng.permutation(full + loose):
        lo = 16 * int(rng.integers(0, 30))
        for _ in range(2):
            inside = np.sort(rng.choice(160, 128 if k < full else 78, replace=False))
            inside[[0, -1]] = 0, 159
            rows += [lo + np.unique(inside)] * 8
    _check(engine_factory, rows, N, K, rng, panels=2 * (full + loose) if panels else 0,
           mfma_tiles=0 if panels else 10 * (full + loose))


@pytest.mark.parametrize("K,groups", [(32, 3), (32, 700), (256, 40)])
def test_panel_lists_cut_for_the_chip(engine_factory, K, groups):
    """Lists of 1 .. 1 300 columns in as many panels as leave the chip idle, nearly fill it, or do."""
    rng = np.random.default_rng(groups)
    N, rows = 5000, []
    for length in rng.choice([16, 17, 63, 64, 65, 127, 129, 200, 511, 513, 1300] if groups < 100 else [40, 65, 130], groups):
        rows += [np.sort(rng.choice(N, int(length), replace=False))] * 8
    _check(engine_factory, rows, N, K, rng, panels=groups)


@pytest.mark.parametrize("N,width", [(60000, 7000), (60000, 6144), (9000, 7000)])
def test_gathered_pairs_wider_than_the_masks(engine_factory, N, width):
    """Near-dense rows over more tile columns than k_gathered_tiles has masks for; N = 60 000 leaves no room for the kept
    bitmaps of the pairs, N = 9 000 does."""
    rng = np.random.default_rng(width + N)
    rows = []
    for i in range(100):
        rows.append(1000 + np.unique(np.concatenate([[0, width - 1], np.flatnonzero(rng.random(width) < 0.62)])))
        rows.append(np.sort(rng.choice(N, int(rng.integers(0, 9)), replace=False)))
    st = _check(engine_factory, rows, N, 32, rng)
    assert st.mfma_tiles >= 6 * ((width + 15) // 16) and st.panels == 0


def test_classifiers_of_many_rows(engine_factory):
    """More 16-row strips than workgroups of the classifiers: tiles, panels, near-dense and short rows among empty ones."""
    rng = np.random.default_rng(3)
    M, N = 1_100_007, 2000
    empty = np.zeros(0, np.int64)
    rows = [empty] * M
    for s in rng.choice(M // 16, 300, replace=False):
        lo, kind = 16 * int(rng.integers(0, 100)), int(rng.integers(0, 3))
        own = [lo + np.arange(48)] * 16 if kind == 0 else [np.sort(rng.choice(N, 60, replace=False))] * 8 + [empty] * 8
        if kind == 2:
            own = [lo + np.flatnonzero(rng.random(200) < 0.6)] + [rng.choice(N, 3, replace=False) for _ in range(15)]
            own = [np.sort(r) for r in own]
        rows[16 * s:16 * s + 16] = own
    rows[M - 7:] = [np.arange(100, 148)] * 7
    st = _check(engine_factory, rows, N, 16, rng)
    assert st.mfma_tiles >= 150 and st.panels >= 50 and st.nnz_short > 0


@pytest.mark.parametrize("near", [False, True])
def test_ragged_tiles_where_columns_are_near(engine_factory, near):
    """Rows of no whole number of 64-byte steps: looked at for tiles only where neighbours tend to share a tile."""
    rng = np.random.default_rng(11)
    N, rows = 40000, []
    for i in range(4000):
        lo = 16 * int(rng.integers(0, N // 16 - 8))
        rows.append(lo + np.arange(80) if near else np.sort(rng.choice(N, 80, replace=False)))
    rows[:64] = [np.arange(256)] * 64
    st = _check(engine_factory, rows, N, 75, rng)
    assert (st.mfma_tiles > 0) == near


@pytest.mark.parametrize("strips,per_strip", [(64, 1), (255, 128), (257, 128), (600, 64)])
def test_window_order_by_one_workgroup_and_by_many(engine_factory, monkeypatch, strips, per_strip):
    """The order of the windows over strips and tile columns: up to 8 192 windows one workgroup sorts, above four launches."""
    monkeypatch.setenv("SDDMM_WINDOW_ORDER", "1")
    rng = np.random.default_rng(strips)
    N, rows = 16 * 2 * per_strip, []
    for _ in range(strips):
        tc = np.sort(rng.choice(N // 16, per_strip, replace=False))
        c = (tc[:, None] * 16 + np.arange(16)[None, :]).ravel()
        rows += [c[(np.arange(len(c)) + r) % 2 == 0] for r in range(16)]
    _check(engine_factory, rows, N, 32, rng, mfma_tiles=strips * per_strip)


@pytest.mark.parametrize("M", [8, 24, 25, 40])
def test_a_matrix_that_ends_with_half_a_strip_of_a_panel(engine_factory, M):
    """8 rows after the last whole strip: they go the way of the strips that are two panels, unless more rows follow."""
    rng = np.random.default_rng(M)
    N, rows = 640, []
    for _ in range((M + 7) // 8):
        rows += [np.sort(rng.choice(160, 90, replace=False))] * 8
    rows = rows[:M]
    st = _check(engine_factory, rows, N, 32, rng)
    assert st.nnz_panel + st.nnz_mfma >= 90 * (M - 1)
    if M % 16 == 8:
        assert st.mfma_tiles == 0 and st.panels == M // 8


@pytest.mark.parametrize("K,groups,panels", [(200, 60, 0), (200, 170, 170), (512, 170, 0), (100, 60, 60)])
def test_panels_of_long_ragged_rows_need_entries(engine_factory, K, groups, panels):
    """Too few panels of long fp32 rows stay on the gather kernels, with every row classified anew."""
    rng = np.random.default_rng(K + groups)
    N, rows = 4000, []
    for _ in range(groups):
        c = 8 * np.sort(rng.choice(N // 8, 25, replace=False))
        rows += [(c[:, None] + np.arange(8)[None, :]).ravel()] * 8
    _check(engine_factory, rows, N, K, rng, panels=panels, mfma_tiles=0)


@pytest.mark.parametrize("strips,tiles", [(2, 140), (40, 130)])
def test_long_strips_wider_than_the_bitmap(engine_factory, strips, tiles):
    """A workgroup per strip whose columns span more than the bitmap holds: one wavefront merges its rows."""
    rng = np.random.default_rng(tiles)
    N, rows = 600_000, []
    for _ in range(strips):
        tc = np.sort(np.concatenate([[0, N // 16 - 1], 1 + rng.choice(N // 16 - 2, tiles - 2, replace=False)]))
        rows += [(tc[:, None] * 16 + np.arange(16)[None, :]).ravel()[(np.arange(16 * tiles) + r) % 9 != 0] for r in range(16)]
    _check(engine_factory, rows, N, 16, rng, mfma_tiles=strips * tiles)

@pytest.mark.parametrize("K", [32, 64, 128])
def test_window_order_with_gathered_pairs(engine_factory, monkeypatch, K):
    """An order asked for by name also where two windows of a gathered pair would share a wavefront: every window once."""
    monkeypatch.setenv("SDDMM_WINDOW_ORDER", "1")
    rng = np.random.default_rng(K)
    N, rows = 3000, []
    for i in range(600):
        lo = int(rng.integers(0, N - 400))
        rows.append(lo + np.flatnonzero(rng.random(400) < 0.5))
        rows += [np.sort(rng.choice(N, 9, replace=False))] * 2
    rows = [16 * s + np.arange(128) for s in range(40) for _ in range(16)] + rows          # 320 tiles of strips before them
    st = _check(engine_factory, rows, N, K, rng)
    assert st.mfma_tiles > 1000


@pytest.mark.parametrize("per_tile,K,dtype,panels", [(160, 64, capi.F32, True), (176, 64, capi.F32, False), (176, 256, capi.F32, False),
                                                     (160, 256, capi.F32, True), (176, 32, capi.F32, True), (192, 32, capi.F32, False),
                                                     (160, 512, capi.BF16, False), (112, 512, capi.BF16, False), (112, 32, capi.BF16, True),
                                                     (112, 300, capi.F32, False), (160, 600, capi.BF16, False)])
def test_strips_of_two_panels_without_a_mixture(engine_factory, monkeypatch, per_tile, K, dtype, panels):
    """Every strip holds the same number of entries per tile: the line that decides for a mixture decides here too."""
    monkeypatch.setenv("SDDMM_LONG_TILES", "1")
    rng = np.random.default_rng(per_tile + K)
    N, rows = 640, []
    for _ in range(40):
        lo = int(rng.integers(0, 30))
        for _ in range(2):
            rows += [np.concatenate([16 * (lo + t) + np.sort(rng.choice(16, per_tile // 16, replace=False)) for t in range(10)])] * 8
    _check(engine_factory, rows, N, K, rng, dtype, panels=80 if panels else 0, mfma_tiles=0 if panels else 400)


@pytest.mark.parametrize("K,near", [(75, False), (75, True), (90, False), (90, True), (300, True)])
def test_sorted_coo_entries_are_looked_at_like_csr(engine_factory, near, K):
    """The same matrix as row-sorted COO: rows of any length go to the tiles only where neighbours tend to share one."""
    rng = np.random.default_rng(12)
    N, rows = 40000, []
    for i in range(4000):
        lo = 16 * (i // 16)
        rows.append(lo + np.arange(80) if near else np.sort(rng.choice(N, 80, replace=False)))
    rows[:64] = [np.arange(256)] * 64
    both = [_check(engine_factory, rows, N, K, np.random.default_rng(1), coo=coo) for coo in (False, True)]
    assert (both[0].mfma_tiles, both[0].panels) == (both[1].mfma_tiles, both[1].panels)
    assert (both[1].mfma_tiles > 0) == near


@pytest.mark.parametrize("kind,K,looked", [("tiles", 15, False), ("tiles", 33, False), ("tiles", 75, True), ("tiles", 100, True),
                                           ("panels", 300, True), ("panels", 512, False), ("tiles", 512, True), ("near-dense", 75, False)])
def test_rows_of_any_length_are_looked_at_where_launches_pay(engine_factory, kind, K, looked):
    """Structured rows of no whole number of steps: short rows and few entries stay on the gather kernels, since a plan that
    looks at them costs more than several launches gain; longer rows do not."""
    rng = np.random.default_rng(K)
    N, rows = 4000, []
    if kind == "tiles":                                          # 338 688 entries
        for _ in range(42):
            rows += [(16 * np.sort(rng.choice(N // 16, 36, replace=False))[:, None] + np.arange(16)[None, :]).ravel()[:504]] * 16
    elif kind == "panels":                                       # 272 000
        for _ in range(170):
            rows += [(8 * np.sort(rng.choice(N // 8, 25, replace=False))[:, None] + np.arange(8)[None, :]).ravel()] * 8
    else:                                                        # 0.83 M, most of them in 1 400 near-dense rows
        for i in range(9400):
            lo = int(rng.integers(0, N - 1385))
            rows.append(lo + np.flatnonzero(rng.random(1385) < 0.4) if i % 7 == 0 else np.sort(rng.choice(N, 9, replace=False)))
    M = len(rows)
    rowptr, col = _csr(rows)
    val = rng.uniform(-1, 1, len(col)).astype(f32)
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    e = engine_factory()
    e.set_dense(A, B)
    e.set_csr(M, N, rowptr, col, val)
    e.plan(capi.AUTO)
    st = e.stats()
    assert (st.mfma_tiles + st.panels > 0) == looked, (len(col), st.mfma_tiles, st.panels)
    e.run()
    ok, worst, i = O.check_values(e.values(), O.sddmm_csr(rowptr, col, val, A, B, threads=0), mag=O.sddmm_csr_f64(rowptr, col, val, A, B)[1])
    assert ok, (i, worst)
    e.close()


@pytest.mark.parametrize("K,dtype", [(512, capi.BF16), (64, capi.F32)])
def test_strips_among_panels_go_with_them(engine_factory, K, dtype):
    """Strips that are two panels, which would be tiles by themselves, next to panels that are not: one launch."""
    rng = np.random.default_rng(K)
    N, rows = 3000, []
    for i in range(60):
        lo = int(rng.integers(0, 160))
        for _ in range(2):
            rows += [np.concatenate([16 * (lo + t) + np.sort(rng.choice(16, 11, replace=False)) for t in range(10)])] * 8
        rows += [np.sort(rng.choice(N, 110, replace=False))] * 8 + [np.sort(rng.choice(N, 110, replace=False))] * 8
    _check(engine_factory, rows, N, K, rng, dtype, panels=240, mfma_tiles=0)
