"""COO -> CSR where the rows are short: row lengths around the limit of the
ranking path, a long row among short ones, duplicates, columns written over the
input columns.  Bit-identical to a stable numpy sort by (row, column)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = {
    "around the limit": [0, 1, 3, 4, 5, 63, 64, 65, 1023, 1024] + [7] * 50,
    "one row over the limit": [1025] + [9] * 100,
    "one long row": [5] * 4000 + [3000] + [5] * 4000,
    "empty rows": [0] * 300 + [40] + [0] * 300,
}


@pytest.mark.parametrize("case", sorted(LENGTHS))
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("in_place", [False, True])
def test_short_rows(case, dtype, in_place):
    from spc5_amd._lib import check, lib
    from spc5_amd.device import stream_ptr
    from spc5_amd.mm import coo_to_csr
    rng = np.random.default_rng(8)
    lengths = np.array(LENGTHS[case])
    nrows, ncols = len(lengths), 500
    i = np.repeat(np.arange(nrows), lengths).astype(np.int32)
    j = rng.integers(0, ncols, len(i)).astype(np.int32)  # duplicates in the longer rows
    order = rng.permutation(len(i))
    i, j = i[order], j[order]
    v = rng.uniform(-1, 1, len(i))
    di, dj, dv = torch.from_numpy(i).cuda(), torch.from_numpy(j).cuda(), torch.from_numpy(v).cuda().to(dtype)
    if in_place:  # the C entry point without a workspace, columns over the input columns
        rp = torch.empty(nrows + 1, dtype=torch.int32, device="cuda")
        col, val = dj, torch.empty_like(dv)
        check(lib().spc5_hip_coo_to_csr(dv.element_size(), nrows, ncols, len(i), 0, di.data_ptr(), dj.data_ptr(),
                                        dv.data_ptr(), rp.data_ptr(), col.data_ptr(), val.data_ptr(),
                                        stream_ptr()), "spc5_hip_coo_to_csr")
    else:
        rp, col, val = coo_to_csr(di, dj, dv, nrows, ncols)
    want = np.lexsort((j, i))
    assert np.array_equal(rp.cpu().numpy(), np.concatenate([[0], np.cumsum(lengths)]))
    assert np.array_equal(col.cpu().numpy(), j[want])
    assert torch.equal(val.cpu(), torch.from_numpy(v[want]).to(dtype))
