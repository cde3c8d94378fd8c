"""Multi-right-hand-side products at column counts that no lane split divides.

A record's lanes are as many as the chunk's columns need, a 16-byte request may
start at any element and the last one of a row overlaps its neighbour: odd k,
chunks whose tail is narrower, X and Y taken out of wider blocks (rows at odd
offsets), runs shorter than a round of requests and longer.  Reference: numpy in
float64 on the dense matrix; bar: normwise 1e-12 (double), 1e-5 (float), as the
other products' tests (a row's sum is at most 450 products in double)."""
import numpy as np
import pytest
import torch

from matgen import clustered_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 1e-5)])
@pytest.mark.parametrize("r,columns", [(1, False), (2, False), (8, False), (2, True), (4, True), (8, True)])
@pytest.mark.parametrize("x16", (None, False, True))
def test_odd_columns(dtype, tol, r, columns, x16):
    from spc5_amd.device import DeviceMatrix
    rp, col, val = clustered_csr(601, 450, seed=r, dtype=dtype, empty_frac=0.1)
    A = DeviceMatrix.from_csr(*(torch.from_numpy(a).cuda() for a in (rp, col, val)), r, ncols=450)
    A.spmm_columns = columns
    if x16 is not None:
        A.spmm_x16 = x16
    Ad = np.zeros((601, 450))
    for i in range(601):
        Ad[i, col[rp[i]:rp[i + 1]]] = val[rp[i]:rp[i + 1]]
    rng = np.random.default_rng(r)
    for k, kt, shift in ((2, 0, 1), (3, 0, 0), (5, 0, 1), (6, 0, 3), (7, 0, 2), (13, 5, 1), (21, 0, 1), (22, 8, 3),
                         (33, 0, 0), (63, 0, 1), (64, 0, 1), (67, 0, 1), (70, 35, 1)):
        Xw = rng.uniform(-1, 1, (450, k + 4)).astype(dtype)
        Yw = rng.uniform(-1, 1, (601, k + 4)).astype(dtype)
        Y = torch.from_numpy(Yw).cuda()
        A.spmm(torch.from_numpy(Xw).cuda()[:, shift:shift + k], Y[:, shift:shift + k], alpha=1.5, beta=0.5, kt=kt)
        got = Y.cpu().numpy()
        ref = Yw.astype(np.float64)
        ref[:, shift:shift + k] = 1.5 * (Ad @ Xw[:, shift:shift + k].astype(np.float64)) + 0.5 * ref[:, shift:shift + k]
        scale = max(np.abs(Ad).sum(axis=1).max(), 1.0)
        assert np.abs(got - ref).max() / scale <= tol, (k, kt, shift)
        outside = np.r_[0:shift, shift + k:k + 4]
        assert np.array_equal(got[:, outside], Yw[:, outside]), (k, kt, shift)
