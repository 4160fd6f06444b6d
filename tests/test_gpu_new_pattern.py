"""What a new pattern starts from and which of its faults is reported.  All GPU."""
import numpy as np
import pytest

from dphpc_amd import capi

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("nnz", [1, 3, 4, 5, 8, 1023, 4097])
def test_no_entry_is_computed_before_the_first_run(engine_factory, nnz):
    """The results of the pattern before lie in the same memory: around the four entries that a thread clears."""
    rowptr, col = np.array([0, nnz], np.int32), np.arange(nnz, dtype=np.int32)
    A, B = np.ones((1, 8), f32), np.ones((nnz, 8), f32)
    with engine_factory() as e:
        e.set_dense(A, B)
        for fresh in ("csr", "coo"):
            e.set_csr(1, nnz, rowptr, col, np.ones(nnz, f32))
            e.plan(capi.AUTO)
            e.run()
            assert (e.values() == 8.0).all()
            if fresh == "csr":
                e.set_csr(1, nnz, rowptr, col, np.ones(nnz, f32))
            else:
                e.set_coo(1, nnz, np.zeros(nnz, np.int32), col, np.ones(nnz, f32))
            assert (e.values() == 0.0).all(), fresh


@pytest.mark.parametrize("rowptr,col,what", [
    ([0, 2, 1, 3], [0, 1, 2], "rowptr"),
    ([0, 2, 1, 3], [0, 99, 2], "rowptr"),          # both: the columns of a malformed row pointer are not looked at
    ([0, 1, 2, 3], [0, 99, 2], "column"),
])
def test_which_fault_is_reported(engine_factory, rowptr, col, what):
    with engine_factory() as e:
        e.set_dense(np.ones((3, 8), f32), np.ones((5, 8), f32))
        with pytest.raises(capi.SddmmError) as ei:
            e.set_csr(3, 5, np.array(rowptr, np.int32), np.array(col, np.int32), np.ones(3, f32))
        assert ei.value.code == capi.ERR_PATTERN and what in str(ei.value)
        e.set_csr(3, 5, np.array([0, 1, 2, 3], np.int32), np.array([0, 1, 2], np.int32), np.ones(3, f32))
        e.plan(capi.AUTO)
        e.run()
        assert (e.values() == 8.0).all()
