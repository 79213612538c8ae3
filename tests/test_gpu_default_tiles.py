"""The tile size that a matrix is opened with: smaller dictionary tiles only where
they gather few more lines and hold several segments, with the sums of the
16384-element ones."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from mlem_amd import synth

pytestmark = pytest.mark.gpu

WIDE, MID, SMALL = ("dict512", 32), ("dict512", 16), ("dict", 8)


def _random(rows, cols, per_row, seed=3):
    rng = np.random.default_rng(seed)
    rowidx = np.cumsum(rng.integers(0, 2 * per_row + 1, rows)).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = rng.integers(0, cols, el.size)
    el["value"] = rng.random(el.size, dtype=np.float32)
    return rowidx, el


@pytest.mark.parametrize("rows,cols,per_row,fwd,bwd", [
    (60000, 60000, 100, WIDE, WIDE),       # 6M elements, many lines more in smaller tiles
    (200000, 100000, 25, WIDE, WIDE),
    (400000, 1500, 10, MID, WIDE),         # columns of 2700 elements, more than a CU's tiles each
    (50000, 50000, 45, MID, MID),          # 2.2M: few more in 8192, many in 2048
    (5000, 4000, 400, MID, MID),           # rows of 400: five in a tile of 2048
    (10000, 10000, 30, SMALL, SMALL),
    (300, 100000, 40, SMALL, SMALL),
])
def test_random_matrices(rows, cols, per_row, fwd, bwd):
    rowidx, el = _random(rows, cols, per_row)
    x = np.random.default_rng(1).random(cols, dtype=np.float32)
    r = np.random.default_rng(2).random(rows, dtype=np.float32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        assert A.launch() == {"fwd": fwd, "bwd": bwd}
        f, b = M.calcFwProj(A, x), M.calcBkProj(A, r)
        A.set_launch(WIDE, WIDE)
        assert np.array_equal(f, M.calcFwProj(A, x)) and np.array_equal(b, M.calcBkProj(A, r))


@pytest.mark.parametrize("grid,lors,fwd,bwd", [
    ((8, 8, 8), 4096, SMALL, SMALL),
    ((64, 60, 24), 80000, MID, MID),       # 4.9M elements
    ((75, 77, 31), 200003, WIDE, WIDE),    # 15.2M
    ((11, 12, 12), 500000, MID, WIDE),     # 6.6M, columns of 4200 elements
])
def test_lines_of_response(grid, lors, fwd, bwd):
    m = synth.make_matrix(grid, lors, 1001)
    with M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid) as A:
        assert A.launch() == {"fwd": fwd, "bwd": bwd}
