"""The fused call where rows are cut into several work items: O is the same bit for bit in every run, whatever the
length at which rows are cut, with and without room for the pieces.  All GPU.  Same bar as test_gpu_fused.py."""
import numpy as np
import pytest

from dphpc_amd import capi
from oracle import oracle as O
from test_gpu_fused import _check, _rounded

pytestmark = pytest.mark.gpu
f32 = np.float32


def _matrix(rng, N, lens):
    rows = [np.sort(rng.choice(N, int(n), replace=False)) for n in lens]
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return rowptr, np.concatenate(rows).astype(np.int32), rng.uniform(-1, 1, rowptr[-1]).astype(f32)


def _operands(rng, M, N, K, dtype):
    A, B = rng.uniform(-1, 1, (M, K)).astype(f32), rng.uniform(-1, 1, (N, K)).astype(f32)
    return (A, A, B, B) if dtype == capi.F32 else _rounded(A, dtype) + _rounded(B, dtype)


# one, two, three, four, six and eight units per lane, 1 .. 8 lanes per entry
@pytest.mark.parametrize("K,dtype", [(4, capi.F32), (12, capi.F32), (32, capi.F32), (64, capi.F16), (96, capi.F32),
                                     (128, capi.F32), (160, capi.F32), (192, capi.BF16), (256, capi.F32)])
@pytest.mark.parametrize("env", [{}, {"SDDMM_FUSED_SEG": "64"}, {"SDDMM_FUSED_BALANCED": "1"}])
def test_cut_rows_repeat(engine_factory, monkeypatch, K, dtype, env):
    """Rows around the default cuts (256, 512, 1024) and of many pieces, in the first and the last wavefront."""
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    rng = np.random.default_rng(K)
    N = 6000
    lens = np.concatenate([[2048, 256, 257, 3], rng.integers(0, 9, 300), [511, 512, 513, 1024, 1025, 5600, 64, 65, 0],
                           rng.integers(0, 9, 40), [1700, 1]])
    M = len(lens)
    rowptr, col, val = _matrix(rng, N, lens)
    Ah, A, Bh, B = _operands(rng, M + 2, N, K, dtype)
    print("cut rows", K, dtype, env, flush=True)
    with engine_factory() as e:
        e.set_dense(Ah, Bh, dtype)
        e.set_csr(M, N, rowptr, col, val)
        first = _check(e, rowptr, col, val, A, B, "K=%d %s" % (K, env))
        for _ in range(20):
            np.testing.assert_array_equal(e.run_fused(), first)


def test_longer_rows_of_the_operands_under_the_same_items(engine_factory):
    """The pattern stays, K grows: the pieces need more room."""
    rng = np.random.default_rng(2)
    N, lens = 3000, [900, 0, 7, 2900, 300]
    rowptr, col, val = _matrix(rng, N, lens)
    with engine_factory() as e:
        A, _, B, _ = _operands(rng, 5, N, 8, capi.F32)
        e.set_dense(A, B)
        e.set_csr(5, N, rowptr, col, val)
        for K in (8, 200, 16):
            A, _, B, _ = _operands(rng, 5, N, K, capi.F32)
            e.set_dense(A, B)
            _check(e, rowptr, col, val, A, B, "K=%d" % K)


def test_without_room_for_the_pieces(engine_factory, monkeypatch):
    rng = np.random.default_rng(3)
    N, lens = 6000, np.concatenate([[5000, 2], rng.integers(0, 20, 200), [600, 257, 70]])
    rowptr, col, val = _matrix(rng, N, lens)
    A, _, B, _ = _operands(rng, len(lens), N, 64, capi.F32)
    monkeypatch.setenv("SDDMM_SPARE_BYTES", "0")
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_csr(len(lens), N, rowptr, col, val)
        first = _check(e, rowptr, col, val, A, B, "no room")
        np.testing.assert_array_equal(e.run_fused(), first)
        monkeypatch.delenv("SDDMM_SPARE_BYTES")
        e.set_csr(len(lens), N, rowptr, col, val)
        _check(e, rowptr, col, val, A, B, "room again")


def test_room_for_fewer_pieces_only(engine_factory, monkeypatch):
    """25 pieces of 256 entries take 6 400 bytes, 5 of 1 024 take 1 280: the sums are then those of the longer pieces."""
    rng = np.random.default_rng(4)
    N, lens = 6000, np.concatenate([[5000, 2], rng.integers(0, 20, 200), [600, 257, 70]])
    rowptr, col, val = _matrix(rng, N, lens)
    A, _, B, _ = _operands(rng, len(lens), N, 64, capi.F32)
    got = []
    for name, value in (("SDDMM_SPARE_BYTES", "4000"), ("SDDMM_FUSED_SEG", "1024"), ("SDDMM_FUSED_SEG", "256"),
                        ("SDDMM_FUSED_PARTS_MAX", "0"), ("SDDMM_FUSED_PARTS_MAX", "1")):
        with monkeypatch.context() as m, engine_factory() as e:
            m.setenv(name, value)
            e.set_dense(A, B)
            e.set_csr(len(lens), N, rowptr, col, val)
            got.append(_check(e, rowptr, col, val, A, B, name))
    np.testing.assert_array_equal(got[0], got[1])
    assert (got[0] != got[2]).any()
    np.testing.assert_array_equal(got[0], got[3])              # more than 0 MiB is too much, the pieces of 256 fit 1
    np.testing.assert_array_equal(got[2], got[4])


def test_room_after_the_operands_grew(engine_factory, monkeypatch):
    """400 rows of 2 000 entries, planned at K = 8 (100 KiB of pieces), then K = 256 (3.2 MB): above 1 MiB pieces of 1 024."""
    monkeypatch.setenv("SDDMM_FUSED_PARTS_MAX", "1")
    rng = np.random.default_rng(6)
    N, lens = 3000, np.full(400, 2000)
    rowptr, col, val = _matrix(rng, N, lens)
    got = []
    for grow in (True, False):
        with engine_factory() as e:
            if grow:
                e.set_dense(*[np.ones((n, 8), f32) for n in (400, N)])
                e.set_csr(400, N, rowptr, col, val)
                e.run_fused()
            else:
                monkeypatch.setenv("SDDMM_FUSED_SEG", "1024")
            A, _, B, _ = _operands(np.random.default_rng(7), 400, N, 256, capi.F32)
            e.set_dense(A, B)
            if not grow:
                e.set_csr(400, N, rowptr, col, val)
            got.append(_check(e, rowptr, col, val, A, B, str(grow)))
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("panel_rows,longer", [(0, 3), (0, 1100), (256, 0)])
def test_a_few_longer_rows_do_not_cut_the_others(engine_factory, monkeypatch, panel_rows, longer):
    """3 600 rows of about 380 entries stay whole beside 3 rows of 2 000, and beside 256 rows of 1 100 that the panel
    kernel takes; beside 1 100 rows of 2 000 too (they are three quarters of the items).  The sums of a row tell whether
    it was cut."""
    rng = np.random.default_rng(5)
    N, bulk, K = 3000, 3600, 32
    lens = np.concatenate([np.full(panel_rows, 1100), rng.integers(375, 386, bulk), np.full(longer, 2000)]).astype(np.int64)
    rowptr, col, val = _matrix(rng, N, lens)
    for r in range(panel_rows):                                # eight rows on the columns of the first
        a = rowptr[r // 8 * 8]
        col[rowptr[r]:rowptr[r + 1]] = col[a:a + 1100]
    M = len(lens)
    A, _, B, _ = _operands(rng, M, N, K, capi.F32)
    got = {}
    for seg in (None, "4096", "256"):                          # by rule, every row whole, every row cut
        with monkeypatch.context() as m, engine_factory() as e:
            if seg:
                m.setenv("SDDMM_FUSED_SEG", seg)
            e.set_dense(A, B)
            e.set_csr(M, N, rowptr, col, val)
            got[seg] = _check(e, rowptr, col, val, A, B, str(seg))
            assert e.stats().kernels_launched == (3 if panel_rows else 2)
    rows = slice(panel_rows, panel_rows + bulk)
    np.testing.assert_array_equal(got[None][rows], got["4096"][rows])
    assert (got["256"][rows] != got["4096"][rows]).any()
    if longer:
        assert (got[None][panel_rows + bulk:] != got["4096"][panel_rows + bulk:]).any()


@pytest.mark.parametrize("K,dtype", [(16, capi.F32), (64, capi.F32), (96, capi.F32), (100, capi.F32), (128, capi.BF16), (136, capi.F16),
                                     (192, capi.BF16), (192, capi.F32), (256, capi.F32), (256, capi.F16), (256, capi.BF16)])
def test_steps_and_batches_give_the_same(engine_factory, monkeypatch, K, dtype):
    """Both forms of the kernel add in the same order.  Rows around its chunks of 64 entries and their halves and quarters;
    an infinite row of B that no entry names and one that a single row names."""
    rng = np.random.default_rng(K + dtype)
    N = 400
    lens = np.concatenate([np.arange(60, 140), [191, 192, 193, 255, 256, 257, 319, 320, 321, 398, 1]])
    rowptr, col, val = _matrix(rng, N - 2, lens)
    Ah, A, Bh, B = _operands(rng, len(lens), N, K, dtype)
    got = {}
    for steps in ("0", "1"):
        monkeypatch.setenv("SDDMM_FUSED_STEPS", steps)
        with engine_factory() as e:
            e.set_dense(Ah, Bh, dtype)
            e.set_csr(len(lens), N, rowptr, col, val)
            o = _check(e, rowptr, col, val, A, B, "steps " + steps)
            got[steps] = (o, e.values())
            wild = Bh.copy()
            wild[N - 1] = wild[col[-1]] = {capi.F32: np.inf, capi.BF16: 0x7F80, capi.F16: 0x7C00}[dtype]
            e.set_dense(Ah, wild, dtype)
            named = np.array([col[-1] in col[rowptr[r]:rowptr[r + 1]] for r in range(len(lens))])
            o = e.run_fused()
            assert np.isfinite(o[~named]).all() and not np.isfinite(o[named]).all(axis=1).any()
    for a, b in zip(got["0"], got["1"]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("K,dtype", [(4, capi.F32), (12, capi.F32), (64, capi.F16), (100, capi.F32), (160, capi.BF16), (256, capi.F32)])
@pytest.mark.parametrize("env", [{}, {"SDDMM_FUSED_SEG": "64"}, {"SDDMM_FUSED_BALANCED": "1"}])
def test_pieces_added_by_a_kernel_of_their_own(engine_factory, monkeypatch, K, dtype, env):
    monkeypatch.setenv("SDDMM_FUSED_ADD_APART", "1")
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    rng = np.random.default_rng(K)
    N, M = 6000, 350
    lens = rng.integers(0, 9, M)
    lens[[0, 1, 2, 63, 64, 65, 200, M - 1]] = [2048, 256, 257, 513, 5900, 1025, 64, 700]
    rowptr, col, val = _matrix(rng, N, lens)
    Ah, A, Bh, B = _operands(rng, M + 2, N, K, dtype)
    with engine_factory() as e:
        e.set_dense(Ah, Bh, dtype)
        for _ in range(2):                                     # a new pattern in the same blocks
            e.set_csr(M, N, rowptr, col, val)
            first = _check(e, rowptr, col, val, A, B, "K=%d %s" % (K, env))
            assert e.stats().kernels_launched == 3
            for _ in range(5):
                np.testing.assert_array_equal(e.run_fused(), first)


@pytest.mark.parametrize("hubs,length,balanced,apart", [(64, 5000, "1", True), (64, 5000, "0", False), (1, 262144, "0", False),
                                                        (1, 262145, "0", True), (1, 600000, "0", True), (0, 0, "0", False)])
def test_which_kernel_adds_the_pieces(engine_factory, monkeypatch, hubs, length, balanced, apart):
    """More than 1 024 pieces of 256 entries for one wavefront of the kernel of the short rows: it takes 64 rows, or 16 at K = 16."""
    monkeypatch.setenv("SDDMM_FUSED_BALANCED", balanced)
    rng = np.random.default_rng(hubs + 1)
    N = max(6000, length + 10)
    lens = np.concatenate([rng.integers(1, 5, 640), np.full(hubs, length)]).astype(np.int64)
    rowptr, col, val = _matrix(rng, N, lens)
    A, _, B, _ = _operands(rng, len(lens), N, 16, capi.F32)
    with engine_factory() as e:
        e.set_dense(A, B)
        e.set_csr(len(lens), N, rowptr, col, val)
        first = _check(e, rowptr, col, val, A, B, "hubs")
        assert e.stats().kernels_launched == (3 if apart else 2 if hubs else 1)
        np.testing.assert_array_equal(e.run_fused(), first)
