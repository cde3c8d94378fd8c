"""Converter groups of 64 rows: groups that exceed the stage and are converted
in runs of fewer rows, window ends at row boundaries, columns near the largest
index.  Byte-identical to the oracle converter."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def rows_to_csr(rows):
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return rowptr, np.concatenate([*rows, np.zeros(0, np.int64)]).astype(np.int32)


def cases():
    rng = np.random.default_rng(2)
    pick = lambda n, k: np.sort(rng.choice(n, k, replace=False))
    light = lambda n: [pick(3000, 5) for _ in range(n)]
    one = light(700)
    one[70] = np.arange(3000)          # its block-row alone exceeds the stage
    some = light(2000)
    for i in range(128, 192, 9):
        some[i] = pick(3000, 200)      # the group fits in halves or quarters
    return {
        "one heavy row": one,
        "heavy group": some,
        "all heavy": [pick(20000, 400) for _ in range(130)],
        # rows end inside the next row's window, empty rows between
        "touching rows": [np.arange(3) + (i % 7) if i % 5 else np.zeros(0, np.int64) for i in range(200)],
        "largest columns": [np.array([i, 2 ** 31 - 20 + i % 9, 2 ** 31 - 2 - i % 3]) for i in range(130)],
    }


@pytest.mark.parametrize("case", sorted(cases()))
@pytest.mark.parametrize("r", [1, 2, 4, 8])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_groups(case, r, dtype):
    from spc5_amd.device import convert_csr
    rowptr, col = rows_to_csr(cases()[case])
    val = np.random.default_rng(3).uniform(-1, 1, len(col)).astype(dtype)
    bptr, hdr, vout, nb = O.convert(r, rowptr, col, val)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    rs, h, v, got = convert_csr(dev(rowptr), dev(col), dev(val), r)
    assert got == nb
    nbr = (len(rowptr) - 1 + r - 1) // r
    assert np.array_equal(rs.cpu().numpy(), np.asarray(bptr[: nbr + 1], np.int32))
    assert np.array_equal(h.cpu().numpy(), np.asarray(hdr, np.uint8))
    assert np.array_equal(v.cpu().numpy().view(np.uint8), np.ascontiguousarray(vout).view(np.uint8))


@pytest.mark.parametrize("columns", [[4, 3], [5, 5], [-1], [3, -2], [-2, -1, 7], [-(2 ** 31)]])
def test_bad_columns_are_refused(columns):
    from spc5_amd import Spc5Error
    from spc5_amd.device import block_count
    rows = [np.arange(6) for _ in range(100)]
    rows[33] = np.array(columns)
    rowptr, col = rows_to_csr(rows)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for r in (1, 2, 4, 8):
        with pytest.raises(Spc5Error, match="strictly increasing"):
            block_count(dev(rowptr), dev(col), r)
