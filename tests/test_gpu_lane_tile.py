"""The lane-block SpMV tile (one block per lane): matrices whose neighbouring
blocks read neighbouring parts of x, at the sizes where the tile can go wrong.

Reference: A decoded to dense rows on the host and multiplied in float64;
tolerance of the product tests, max|y - y_ref| <= tol max(||A||_inf ||x||_inf,
||y0||_inf) with tol = 1e-12 (double) and 1e-5 (float sums).
"""
import numpy as np
import pytest
import torch

from conftest import normwise_error

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5, "f32v8": 1e-5, "bf16": 1e-5}
VEC = {"f64": torch.float64, "f32": torch.float32, "f32v8": torch.float32, "bf16": torch.float32}


def csr(n, ncols, rows_of, seed):
    """CSR with the columns rows_of(i) (clipped to the matrix) and values U[-1,1]."""
    rng = np.random.default_rng(seed)
    cols = [np.unique(np.clip(rows_of(i), 0, ncols - 1)) if len(rows_of(i)) else np.zeros(0, int) for i in range(n)]
    rowptr = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    col = np.concatenate(cols + [np.zeros(0, int)]).astype(np.int32)
    return rowptr, col, rng.uniform(-1, 1, len(col))


def shapes():
    band = lambda i, w: np.arange(i - w, i + w + 1)
    return {
        # x shorter than two windows: every block's window reaches past its end
        "ends": (40, 17, lambda i: np.array([16, 15, 0]) if i % 3 else np.array([16])),
        # rows that do not fill the last block-row, tiles of 64 block-rows +- 1
        "edges": (64 * 8 + 1, 64 * 8 + 1, lambda i: band(i, 2)),
        # runs of empty rows longer than a tile, then rows of many batches
        "gaps": (700, 700, lambda i: band(i, 60) if i % 300 < 3 else np.zeros(0, int)),
        # full blocks: every position set
        "dense": (70, 90, lambda i: np.arange(90)),
        # one long row among short ones
        "long": (300, 3000, lambda i: np.arange(0, 3000, 2) if i == 150 else band(i, 1)),
    }


def matrix(kind, r, rowptr, col, val, ncols, offset):
    """A DeviceMatrix whose headers, values and vectors start `offset` elements into their buffers."""
    from spc5_amd.device import DeviceMatrix, convert_csr
    from spc5_amd.solver import lowp
    dt = torch.float32 if kind == "f32" else torch.float64
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    rs, hdr, v, nb = convert_csr(dev(rowptr), dev(col), dev(val).to(dt), r)

    def moved(t, by):
        buf = torch.zeros(t.numel() + by, dtype=t.dtype, device="cuda")
        buf[by:] = t
        return buf[by:]

    m = DeviceMatrix(r=r, vs=16 if kind == "f32" else 8, nrows=len(rowptr) - 1, ncols=ncols, nnz=len(col), nblocks=nb,
                     rows_size=rs, headers=moved(hdr, 5 * offset), values=moved(v, offset))
    if kind in ("f32v8", "bf16"):
        low = lowp(m, "f32" if kind == "f32v8" else "bf16")
        return m.values_view(moved(low.values, offset))
    return m


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", sorted(shapes()))
@pytest.mark.parametrize("r", [1, 2, 4, 8])
@pytest.mark.parametrize("kind", sorted(TOL))
def test_lane_tile(kind, r, shape, offset):
    from spc5_amd.batch import Batch
    from spc5_amd.solver import spmv_ex
    n, ncols, rows_of = shapes()[shape]
    rowptr, col, val = csr(n, ncols, rows_of, 3)
    if kind == "bf16":
        val = torch.from_numpy(val).float().bfloat16().double().numpy()
    elif kind != "f64":
        val = val.astype(np.float32).astype(np.float64)
    m = matrix(kind, r, rowptr, col, val, ncols, offset)
    rng = np.random.default_rng(5)
    vec = lambda k: torch.from_numpy(rng.uniform(-1, 1, k + offset)).cuda().to(VEC[kind])[offset:]
    x, y0 = vec(ncols), vec(n)
    xh, y0h = x.double().cpu().numpy(), y0.double().cpu().numpy()
    ax = np.zeros(n)
    np.add.at(ax, np.repeat(np.arange(n), np.diff(rowptr)), val * xh[col])

    def check(y, want, scale):
        err = normwise_error(y.double().cpu().numpy(), want, rowptr, val * scale, xh, y0h)
        assert err <= TOL[kind], err

    for tile_values in (0, 64, 1 << 20):
        m.tile_values = tile_values
        check(m.spmv(x, y0.clone()), y0h + ax, 1.0)
    check(spmv_ex(m, x, torch.full_like(y0, float("nan")), alpha=-2.0, beta=0.0), -2.0 * ax, 2.0)
    check(spmv_ex(m, x, y0.clone(), alpha=0.5, beta=-1.5), 0.5 * ax - 1.5 * y0h, 1.0)
    # two of them in one batch: the same tile, the same bits
    ya, yb, y1 = y0.clone(), torch.zeros_like(y0), m.spmv(x, y0.clone())
    Batch([m, m], [x, x], [ya, yb]).spmv()
    assert torch.equal(ya, y1)
    check(yb, ax, 1.0)


@pytest.mark.parametrize("kind", sorted(TOL))
def test_lane_tile_keeps_infinities_apart(kind):
    """An infinite x entry reaches the rows that use its column and no other."""
    n = 200
    rowptr, col, val = csr(n, n, lambda i: np.array([i - 1, i, i + 3]), 4)
    m = matrix(kind, 2, rowptr, col, val, n, 0)
    x = torch.ones(n, dtype=VEC[kind], device="cuda")
    x[77] = float("inf")
    y = m.spmv(x, torch.zeros_like(x)).cpu().numpy()
    hit = np.zeros(n, bool)
    hit[np.repeat(np.arange(n), np.diff(rowptr))[col == 77]] = True
    assert np.array_equal(np.isinf(y), hit) and not np.isnan(y).any()


def test_batch_of_both_tiles_and_every_r():
    """Local and scattered matrices of different r share one launch; each y
    is bit-identical to its matrix's own product."""
    from spc5_amd.batch import Batch
    from spc5_amd.device import DeviceMatrix
    rng = np.random.default_rng(9)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    mats, xs = [], []
    for k, r in enumerate((1, 2, 4, 8, 4, 8)):
        n = 3000 + 17 * k
        spread = k >= 4
        rowptr, col, val = csr(n, n, lambda i: rng.integers(0, n, 12) if spread else np.arange(i - 4, i + 5), k)
        mats.append(DeviceMatrix.from_csr(dev(rowptr), dev(col), dev(val), r))
        xs.append(dev(rng.uniform(-1, 1, n)))
    ys = [torch.ones_like(x) for x in xs]
    want = [m.spmv(x, torch.ones_like(x)) for m, x in zip(mats, xs)]
    Batch(mats, xs, ys).spmv()
    for a, b in zip(ys, want):
        assert torch.equal(a, b)
