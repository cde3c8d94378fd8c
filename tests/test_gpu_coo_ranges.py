"""COO -> CSR of many entries, whose rows are counted in ranges of 32,768 rows and
chunks of entries: row counts at the edges of a range, chunks with a remainder,
duplicates, a row too long, rows and columns out of range.  Bit-identical to a
stable numpy sort by (row, column)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def entries(nrows, nnz, order, seed=3):
    rng = np.random.default_rng(seed)
    i = np.r_[rng.integers(0, nrows, nnz - 2), 0, nrows - 1].astype(np.int32)
    if order == "in order":
        i.sort()
    j = rng.integers(0, 700, nnz).astype(np.int32)
    return i, j, rng.uniform(-1, 1, nnz)


@pytest.mark.parametrize("order", ["shuffled", "in order"])
@pytest.mark.parametrize("nrows,nnz", [(2003, 131072), (32767, 140001), (32768, 131073), (32769, 300000),
                                       (65537, 200003), (1048576, 150000), (1048577, 150000)])
def test_ranges(nrows, nnz, order):
    from spc5_amd.mm import coo_to_csr
    i, j, v = entries(nrows, nnz, order)
    rp, col, val = coo_to_csr(*(torch.from_numpy(a).cuda() for a in (i, j, v)), nrows, 700)
    want = np.lexsort((j, i))
    assert np.array_equal(rp.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(i, minlength=nrows))]))
    assert np.array_equal(col.cpu().numpy(), j[want])
    assert np.array_equal(val.cpu().numpy(), v[want])


@pytest.mark.parametrize("length", [1024, 1025, 70000])
def test_long_row(length):
    from spc5_amd.mm import coo_to_csr
    i, j, v = entries(40001, 200000, "shuffled")
    i[:] = np.where(i == 33333, 5, i)
    i[1000:1000 + length] = 33333
    rp, col, val = coo_to_csr(*(torch.from_numpy(a).cuda() for a in (i, j, v)), 40001, 700)
    want = np.lexsort((j, i))
    assert np.array_equal(rp.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(i, minlength=40001))]))
    assert np.array_equal(col.cpu().numpy(), j[want]) and np.array_equal(val.cpu().numpy(), v[want])


@pytest.mark.parametrize("what,value", [("row", -1), ("row", 40001), ("column", -1), ("column", 700)])
def test_out_of_range(what, value):
    from spc5_amd._lib import Spc5Error
    from spc5_amd.mm import coo_to_csr
    i, j, v = entries(40001, 200000, "shuffled")
    (i if what == "row" else j)[77777] = value
    with pytest.raises(Spc5Error, match="out of range"):
        coo_to_csr(*(torch.from_numpy(a).cuda() for a in (i, j, v)), 40001, 700)
