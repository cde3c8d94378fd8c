"""Performance cases: the work a program built on this library has it do.

Every case starts from a matrix made on the GPU with plain torch and goes
through the public Python entry points (DeviceMatrix, Batch, coo_to_csr,
solver).  A case's sizes fix its sparsity pattern; the seed gives the values,
the vectors and the order of the triplets.  The matrix families are the ones the benchmark and the tests use:
the 5-point Laplacian, the 27-point stencil, clustered runs (lognormal row
lengths, runs of 1..16 columns near the diagonal) and banded matrices with
30 % of the band filled.

`kind` says which path a case takes:

* spmv      y += A x, the product a program repeats thousands of times
* spmm      Y = alpha A X + beta Y for k right-hand sides
* batch     y_i += A_i x_i for many uneven matrices in one graph launch
* convert   CSR -> beta(r,VS) with its plan (DeviceMatrix.from_csr)
* assemble  unsorted COO -> CSR -> beta(r,VS)
* cg        conjugate gradient in double
* mixed_cg  conjugate gradient on float values with double residuals
"""
from __future__ import annotations

import math

import torch

from spc5_amd.batch import Batch
from spc5_amd.device import DeviceMatrix
from spc5_amd.mm import coo_to_csr
from spc5_amd.solver import cg, lowp, mixed_cg

_FAMILIES = ("lap2d", "stencil27", "clustered", "banded")


def listed():
    return [
        # a small grid problem: one launch, where latency is all there is
        {"name": "spmv f64 laplacian 64^2", "kind": "spmv", "family": "lap2d", "n": 64, "type": "f64", "r": 4},
        # a grid that fits the caches, odd edge: short rows, the conversion's
        # default one row per block
        {"name": "spmv f64 laplacian 511^2", "kind": "spmv", "family": "lap2d", "n": 511, "type": "f64", "r": 1},
        # the benchmark's headline product: 4 M rows, far larger than the caches
        {"name": "spmv f64 clustered 4M", "kind": "spmv", "family": "clustered", "n": 4194304, "type": "f64", "r": 1},
        # a float matrix in the reference's float format (16-column blocks), odd size
        {"name": "spmv f32 clustered 1M", "kind": "spmv", "family": "clustered", "n": 1000003, "type": "f32", "r": 2},
        # the reduced-precision copy of a double stencil matrix, row-sorted as
        # the solve benchmark chooses
        {"name": "spmv bf16 stencil 128^3", "kind": "spmv", "family": "stencil27", "n": 128, "type": "bf16", "r": 2,
         "row_sort": True},
        # block Krylov / many load cases: the widest column chunk in double
        {"name": "spmm f64 stencil 96^3 k64", "kind": "spmm", "family": "stencil27", "n": 96, "type": "f64", "r": 4,
         "k": 64, "columns": True},
        # a few right-hand sides, an odd count, default options
        {"name": "spmm f32 clustered 300k k5", "kind": "spmm", "family": "clustered", "n": 300007, "type": "f32",
         "r": 2, "k": 5, "columns": False},
        # many uneven systems at once (rows 1,000 .. 200,000, bandwidths 4 .. 256)
        {"name": "batch f64 96 banded", "kind": "batch", "count": 96, "type": "f64", "r": 4},
        # a large matrix entering the format
        {"name": "convert f64 clustered 1M", "kind": "convert", "family": "clustered", "n": 1048576, "type": "f64",
         "r": 4},
        # a file's worth of unsorted float triplets up to a matrix ready to multiply
        {"name": "assemble f32 banded 50k", "kind": "assemble", "family": "banded", "n": 50021, "bw": 40,
         "type": "f32", "r": 1},
        # a small solve, bound by launches and reductions
        {"name": "cg f64 stencil 24^3", "kind": "cg", "family": "stencil27", "n": 24, "type": "f64", "r": 1,
         "rtol": 1e-12},
        # the precision form: float iteration, double residuals
        {"name": "mixed cg f32 stencil 96^3", "kind": "mixed_cg", "family": "stencil27", "n": 96, "type": "f32",
         "r": 2, "row_sort": True, "rtol": 1e-12},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_size(rng, family, rows):
    """Grid edge (laplacian, stencil) or rows (clustered, banded), at most `rows` rows."""
    n = _log_int(rng, 4096, rows)
    if family == "lap2d":
        return {"n": max(16, math.isqrt(n))}
    if family == "stencil27":
        return {"n": max(8, int(round(n ** (1 / 3))) - 1)}
    if family == "banded":
        return {"n": max(1000, n // 4), "bw": rng.randint(4, 128)}
    return {"n": n}


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "spmm", "spmm", "batch", "convert", "convert", "assemble", "cg",
                       "mixed_cg"])
    r = rng.choice([1, 2, 4, 8])
    if kind == "batch":
        return {"kind": kind, "count": _log_int(rng, 4, 80), "type": rng.choice(["f64", "f32"]), "r": r}
    if kind in ("cg", "mixed_cg"):
        n = rng.randint(12, 40) if kind == "cg" else rng.randint(32, 90)
        return {"kind": kind, "family": "stencil27", "n": n, "type": "f64" if kind == "cg" else "f32",
                "r": rng.choice([1, 2]), "row_sort": rng.random() < 0.5, "rtol": 1e-12}
    family = rng.choice(_FAMILIES)
    if kind == "assemble":
        return {"kind": kind, "family": family, **_draw_size(rng, family, 100000), "type": rng.choice(["f64", "f32"]),
                "r": r}
    if kind == "convert":
        return {"kind": kind, "family": family, **_draw_size(rng, family, 1000000),
                "type": rng.choice(["f64", "f64", "f32"]), "r": r}
    case = {"kind": kind, "family": family, "type": rng.choice(["f64", "f64", "f32", "f32", "bf16"]), "r": r}
    if kind == "spmv":
        case.update(_draw_size(rng, family, 2000000), row_sort=r in (2, 4) and rng.random() < 0.3)
    else:
        case.update(_draw_size(rng, family, 300000), k=_log_int(rng, 2, 64), columns=r > 1 and rng.random() < 0.5)
    return case


# ---- matrices ---------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _pattern_generator(n):
    return _generator(1000003 + n)


def _uniform(n, g, lo=-1.0, hi=1.0):
    return torch.rand(n, dtype=torch.float64, device="cuda", generator=g) * (hi - lo) + lo


def _csr_from_mask(keep, cols):
    """Row pointers and columns of the kept entries of a (rows x candidates) table, columns ascending."""
    counts = keep.sum(1)
    rowptr = torch.zeros(keep.shape[0] + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(counts, 0)
    return rowptr.to(torch.int32), cols[keep].to(torch.int32)


def _grid(n, dims, offsets):
    """Structure of a stencil on an n^dims grid and the index of every entry's offset."""
    rows = torch.arange(n ** dims, device="cuda")
    at = [(rows // n ** d) % n for d in range(dims)]  # coordinates, fastest first
    keep, cols = [], []
    for o in offsets:
        ok = torch.ones_like(rows, dtype=torch.bool)
        for d in range(dims):
            ok &= (at[d] + o[d] >= 0) & (at[d] + o[d] < n)
        keep.append(ok)
        cols.append(rows + sum(o[d] * n ** d for d in range(dims)))
    rowptr, col = _csr_from_mask(torch.stack(keep, 1), torch.stack(cols, 1))
    return rowptr, col


def _row_index(rowptr, nnz):
    n = rowptr.numel() - 1
    counts = (rowptr[1:] - rowptr[:-1]).to(torch.int64)
    return torch.repeat_interleave(torch.arange(n, device="cuda"), counts, output_size=nnz)


def _stencil_matrix(family, n, g, constant):
    if family == "lap2d":
        offsets = [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)]
        rowptr, col = _grid(n, 2, offsets)
        diag = 4.0
    else:
        offsets = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
        rowptr, col = _grid(n, 3, offsets)
        diag = 26.001
    nnz = col.numel()
    # constant coefficients for the solves, a varying medium for the products
    val = torch.full((nnz,), -1.0, dtype=torch.float64, device="cuda") if constant else -_uniform(nnz, g, 0.5, 1.5)
    val[_row_index(rowptr, nnz) == col] = diag
    return rowptr, col, val


def _clustered_matrix(n, g):
    p = _pattern_generator(n)
    length = torch.exp(torch.randn(n, dtype=torch.float64, device="cuda", generator=p) * 0.8
                       + (math.log(32.0) - 0.32)).clamp_(1, 512)
    runs = torch.clamp((length / 8.5).round().to(torch.int64), min=1)
    total = int(runs.sum())
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), runs, output_size=total)
    half = max(16, n // 64)
    first = row + torch.randint(-half, half + 1, (total,), device="cuda", generator=p)
    size = torch.randint(1, 17, (total,), device="cuda", generator=p)
    entries = int(size.sum())
    begin = torch.cumsum(size, 0) - size
    run = torch.repeat_interleave(torch.arange(total, device="cuda"), size, output_size=entries)
    c = first[run] + (torch.arange(entries, device="cuda") - begin[run])
    ok = (c >= 0) & (c < n)
    key = torch.unique(row[run][ok] * n + c[ok])  # overlapping runs share entries
    row, col = key // n, (key % n).to(torch.int32)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return rowptr.to(torch.int32), col, _uniform(col.numel(), g)


def _banded_matrix(n, bw, g, fill=0.3):
    offset = torch.arange(-bw, bw + 1, device="cuda")
    cols = torch.arange(n, device="cuda")[:, None] + offset[None, :]
    keep = torch.rand((n, 2 * bw + 1), device="cuda", generator=_pattern_generator(n)) < fill
    keep[:, bw] = True
    keep &= (cols >= 0) & (cols < n)
    rowptr, col = _csr_from_mask(keep, cols)
    val = _uniform(col.numel(), g)
    val[_row_index(rowptr, col.numel()) == col] += float(bw)
    return rowptr, col, val


def _matrix(case, g, constant=False):
    """(rowptr, col, values) on the GPU, int32 / int32 / float64."""
    if case["family"] in ("lap2d", "stencil27"):
        return _stencil_matrix(case["family"], case["n"], g, constant)
    if case["family"] == "banded":
        return _banded_matrix(case["n"], case["bw"], g)
    return _clustered_matrix(case["n"], g)


_DTYPE = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.float32}  # of the vectors


def _rounded(val, type_):
    """The matrix values a case of this type holds."""
    if type_ == "bf16":
        return val.to(torch.float32).to(torch.bfloat16)
    return val.to(_DTYPE[type_])


def _batch_inputs(case, g):
    u = _uniform(2 * case["count"], _pattern_generator(case["count"]), 0.0, 1.0).tolist()
    out = []
    for i in range(case["count"]):
        n, bw = int(round(1000.0 * 200.0 ** u[2 * i])), 4 + int(u[2 * i + 1] * 253.0)
        rowptr, col, val = _banded_matrix(n, bw, g)
        out.append((rowptr, col, _rounded(val, case["type"]), _uniform(n, g).to(_DTYPE[case["type"]])))
    return out


def _solve_inputs(case, g):
    """The matrix, the solution and its right-hand side, the stencil summed one dimension after another."""
    rowptr, col, val = _matrix(case, g, constant=True)
    n = case["n"]
    x = _uniform(n ** 3, g)
    box = x.view(n, n, n)
    for d in range(3):
        side = torch.zeros_like(box.narrow(d, 0, 1))
        padded = torch.cat([side, box, side], d)
        box = padded.narrow(d, 0, n) + padded.narrow(d, 1, n) + padded.narrow(d, 2, n)
    return rowptr, col, val, x, 27.001 * x - box.reshape(-1)


def _inputs(case, g):
    rowptr, col, val = _matrix(case, g)
    return rowptr, col, _rounded(val, case["type"])


def _vectors(case, rows, g):
    """x and y (products), X and Y (several right-hand sides)."""
    dt = _DTYPE[case["type"]]
    if case["kind"] == "spmv":
        return _uniform(rows, g).to(dt), _uniform(rows, g).to(dt)
    k = case["k"]
    return _uniform(rows * k, g).to(dt).view(rows, k), _uniform(rows * k, g).to(dt).view(rows, k)


def _device_matrix(case, rowptr, col, val):
    if case["type"] == "bf16":
        # bfloat16 values belong to a double matrix's block structure
        m = lowp(DeviceMatrix.from_csr(rowptr, col, val.double(), case["r"]), "bf16")
    else:
        m = DeviceMatrix.from_csr(rowptr, col, val, case["r"])
    if case.get("row_sort"):
        m.row_sort = True
    if case.get("columns"):
        m.spmm_columns = True
    return m


# ---- the cases --------------------------------------------------------------


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "batch":
        parts = _batch_inputs(case, g)
        rows = [p[3].numel() for p in parts]
        y = torch.zeros(sum(rows), dtype=_DTYPE[case["type"]], device="cuda")
        mats = [DeviceMatrix.from_csr(rp, c, v, case["r"]) for rp, c, v, _ in parts]
        return {"case": case, "batch": Batch(mats, [p[3] for p in parts], list(torch.split(y, rows))), "y": y}
    if kind in ("cg", "mixed_cg"):
        rowptr, col, val, _, b = _solve_inputs(case, g)
        a = DeviceMatrix.from_csr(rowptr, col, val, case["r"])
        a.row_sort = bool(case.get("row_sort"))
        low = None
        if kind == "mixed_cg":
            low = lowp(a, case["type"])
            low.row_sort = a.row_sort
        return {"case": case, "a": a, "low": low, "b": b}
    rowptr, col, val = _inputs(case, g)
    n = rowptr.numel() - 1
    if kind == "convert":
        return {"case": case, "csr": (rowptr, col, val)}
    if kind == "assemble":
        order = torch.randperm(col.numel(), device="cuda", generator=g)
        i = _row_index(rowptr, col.numel()).to(torch.int32)[order].contiguous()
        return {"case": case, "n": n, "coo": (i, col[order].contiguous(), val[order].contiguous())}
    x, y = _vectors(case, n, g)
    return {"case": case, "a": _device_matrix(case, rowptr, col, val), "x": x, "y": y}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "spmv":
        return state["a"].spmv(state["x"], state["y"])
    if kind == "spmm":
        return state["a"].spmm(state["x"], state["y"], alpha=1.0, beta=0.5)
    if kind == "batch":
        state["batch"].spmv()
        return state["y"]
    if kind == "cg":
        # the solution; the iteration count and the last residual are rounding's
        return cg(state["a"], state["b"], rtol=case["rtol"])[0]
    if kind == "mixed_cg":
        return mixed_cg(state["a"], state["low"], state["b"], rtol=case["rtol"])[0]
    if kind == "convert":
        m = DeviceMatrix.from_csr(*state["csr"], case["r"])
        return {"rows_size": m.rows_size, "headers": m.headers, "values": m.values}
    rowptr, col, val = coo_to_csr(*state["coo"], state["n"], state["n"])
    m = DeviceMatrix.from_csr(rowptr, col, val, case["r"])
    return {"rowptr": rowptr, "col": col, "val": val, "rows_size": m.rows_size, "headers": m.headers,
            "values": m.values}


# ---- what a pass cannot do without, and its exact answer ---------------------


def _iterations(case):
    """About how many steps CG takes: half the bound from the condition number."""
    lo = 27.001 - (1 + 2 * math.cos(math.pi / (case["n"] + 1))) ** 3
    return max(8.0, 0.25 * math.log(2 / case["rtol"]) * math.sqrt(36.0 / lo))


def work(case):
    g = _generator(0)
    kind = case["kind"]
    if kind == "batch":
        mats = [DeviceMatrix.from_csr(rp, c, v, case["r"]) for rp, c, v, _ in _batch_inputs(case, g)]
        return {"bytes": sum(m.algorithmic_bytes() for m in mats), "flops": sum(2 * m.nnz for m in mats)}
    if kind in ("cg", "mixed_cg"):
        rowptr, col, val = _matrix(case, g, constant=True)
        m = DeviceMatrix.from_csr(rowptr, col, val, case["r"])
        size = 8 if kind == "cg" else 4
        its, n = _iterations(case), m.nrows
        # per step: the matrix, q = A p with p.q, the residual with its norm, x and p
        matrix = m.nnz * size + m.nblocks * m.header_bytes() + 4 * m.info()["nblockrows"]
        return {"bytes": its * (matrix + 10 * n * size), "flops": its * (2 * m.nnz + 10 * n)}
    rowptr, col, val = _inputs(case, g)
    n, nnz, size = rowptr.numel() - 1, col.numel(), val.element_size()
    if kind in ("spmv", "spmm"):
        m = _device_matrix(case, rowptr, col, val)
        k = case.get("k", 1)
        vectors = 3 * n * m.vec_dtype.itemsize
        return {"bytes": m.algorithmic_bytes() + (k - 1) * vectors, "flops": 2 * nnz * k}
    m = DeviceMatrix.from_csr(rowptr, col, val, case["r"])
    made = nnz * size + m.nblocks * m.header_bytes() + 4 * m.info()["nblockrows"]
    csr = 4 * n + nnz * (4 + size)
    return {"bytes": made + csr + ((8 + size) * nnz if kind == "assemble" else 0), "flops": 0}


def _product(rowptr, col, val, x, columns=8):
    """A x or A X in double, X a few columns at a time."""
    row, c = _row_index(rowptr, col.numel()), col.to(torch.int64)
    val, x = val.double(), x.double()
    out = torch.zeros((rowptr.numel() - 1, *x.shape[1:]), dtype=torch.float64, device="cuda")
    if x.dim() == 1:
        return out.index_add_(0, row, val * x[c])
    for j in range(0, x.shape[1], columns):
        part = x[:, j:j + columns].contiguous()
        out[:, j:j + columns] = torch.zeros_like(part).index_add_(0, row, val[:, None] * part[c])
    return out


def exact(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("convert", "assemble"):
        return None  # bytes, whole numbers and moved values: nothing is rounded
    if kind == "batch":
        return torch.cat([_product(rp, c, v, x) for rp, c, v, x in _batch_inputs(case, g)])
    if kind in ("cg", "mixed_cg"):
        return _solve_inputs(case, g)[3]
    rowptr, col, val = _inputs(case, g)
    x, y = _vectors(case, rowptr.numel() - 1, g)
    return _product(rowptr, col, val, x) + (1.0 if kind == "spmv" else 0.5) * y.double()
