"""Products whose blocks are dense enough for a larger stage of the lane-block
tile: double beta(4,8) from 8 and from 10 values a block, float beta(8,16) from 16,
up to full blocks, and batches of matrices on different levels (bit-identical to
each matrix's own product).  Reference: numpy in float64; a row's sum of at most
64 products stays within 64 x 2^-53 (double) or 64 x 2^-24 (float) of the sum of
its products' magnitudes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def banded(n, width, fill, dtype, seed):
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(n):
        lo = max(0, min(i // 8 * 8, n - width))
        c = lo + np.flatnonzero(rng.random(width) < fill)
        rows.append(len(c))
        cols.append(c)
    rp = np.r_[0, np.cumsum(rows)].astype(np.int32)
    col = np.concatenate(cols).astype(np.int32)
    return rp, col, rng.uniform(-1, 1, len(col)).astype(dtype)


def reference(rp, col, val, x):
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    p = val.astype(np.float64) * x.astype(np.float64)[col]
    n = len(rp) - 1
    return np.bincount(row, p, n), np.bincount(row, np.abs(p), n)


FILLS = (0.1, 0.27, 0.33, 0.5, 1.0)


@pytest.mark.parametrize("dtype,r,eps", [(np.float64, 4, 2.0**-53), (np.float32, 8, 2.0**-24)])
def test_levels(dtype, r, eps):
    from spc5_amd.batch import Batch
    from spc5_amd.device import DeviceMatrix
    dev = lambda a: torch.from_numpy(a).cuda()
    mats, xs, ys, own = [], [], [], []
    for k, (n, fill) in enumerate((n, f) for n in (77, 3001) for f in FILLS):
        rp, col, val = banded(n, 64, fill, dtype, k)
        m = DeviceMatrix.from_csr(dev(rp), dev(col), dev(val), r, ncols=n)
        x = np.random.default_rng(k).uniform(-1, 1, n).astype(dtype)
        y = torch.zeros(n, dtype=m.vec_dtype, device="cuda")
        m.spmv(dev(x), y)
        want, size = reference(rp, col, val, x)
        assert np.all(np.abs(y.cpu().numpy() - want) <= 64 * eps * size), (n, fill)
        mats.append(m)
        xs.append(dev(x))
        ys.append(torch.zeros_like(y))
        own.append(y)
    b = Batch(mats, xs, ys)
    b.spmv()
    torch.cuda.synchronize()
    for y, o in zip(ys, own):
        assert torch.equal(y, o)
