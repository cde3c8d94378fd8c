"""The vector kernels of the conjugate gradient iteration at their edges: fewer
elements than a 16-byte request, remainders, more elements than one round of the
grid, x at an odd offset, and products of more and fewer tiles than one kernel
sums by itself.  A tridiagonal system (diagonal 4, neighbours -1; eigenvalues in
(2, 6), condition below 3) solved to a relative residual of 1e-10 (double) or
1e-5 (float) is within 3 times that of the direct solution, plus rounding: 1e-9
and 1e-4."""
import numpy as np
import pytest
import scipy.linalg
import torch

pytestmark = pytest.mark.gpu


def tridiagonal(n, dtype):
    i = np.arange(n)
    counts = np.full(n, 3)
    counts[0] -= 1
    counts[-1] -= 1
    rp = np.r_[0, np.cumsum(counts)].astype(np.int32)
    col = (i[:, None] + np.array([-1, 0, 1])).ravel()
    val = np.broadcast_to(np.array([-1.0, 4.0, -1.0]), (n, 3)).ravel()
    ok = (col >= 0) & (col < n)
    return rp, col[ok].astype(np.int32), val[ok].astype(dtype)


@pytest.mark.parametrize("dtype,rtol,tol", [(np.float64, 1e-10, 1e-9), (np.float32, 1e-5, 1e-4)])
@pytest.mark.parametrize("n,tile", [(1, 0), (2, 0), (3, 0), (5, 0), (1023, 0), (1026, 0), (524291, 0), (600001, 64)])
def test_tridiagonal(dtype, rtol, tol, n, tile):
    from spc5_amd.device import DeviceMatrix
    from spc5_amd.solver import cg
    rp, col, val = tridiagonal(n, dtype)
    A = DeviceMatrix.from_csr(*(torch.from_numpy(a).cuda() for a in (rp, col, val)), 1, ncols=n)
    if tile:
        A.tile_values = tile  # 3 tiles per 64 rows: 28,000
    b = np.random.default_rng(n).uniform(-1, 1, n).astype(dtype)
    wide = torch.zeros(n + 3, dtype=torch.float64 if dtype == np.float64 else torch.float32, device="cuda")
    x, stats = cg(A, torch.from_numpy(b).cuda(), x=wide[1:n + 1], rtol=rtol,
                  maxit=min(n, 200))  # never past an exactly solved system
    ab = np.zeros((3, n))
    ab[0, 1:] = ab[2, :-1] = -1.0
    ab[1] = 4.0
    ref = scipy.linalg.solve_banded((1, 1), ab, b.astype(np.float64)) if n > 1 else b.astype(np.float64) / 4.0
    assert stats["relres"] <= 10 * rtol
    assert np.linalg.norm(x.cpu().numpy() - ref) <= tol * np.linalg.norm(ref)
    assert wide[0].item() == 0.0 and not wide[n + 1:].any()
